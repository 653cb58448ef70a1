"""A masked reset allocates nothing: what it stages the environment ids in comes with the world."""
import pytest

from conftest import nk

pytestmark = pytest.mark.gpu


def mapped_kilobytes():
    with open("/proc/self/status") as status:
        return next(int(line.split()[1]) for line in status if line.startswith("VmSize:"))


def test_the_first_masked_reset_of_a_world_allocates_nothing(device):
    E = 1 << 18                                     # ids of as many environments are a megabyte
    cfg = nk.synthetic.config(1, 8)
    desc = nk.abi.world_desc(E, cfg.dt)
    used, fresh = (nk.World(device, cfg.template, desc) for _ in range(2))
    for _ in range(2):                              # what the runtime itself sets up for a first copy and launch
        used.reset_envs([5, 0, 5])
    before = mapped_kilobytes()
    fresh.reset_envs([7, E - 1, 7])
    assert mapped_kilobytes() - before < 512
    used.close(); fresh.close()
