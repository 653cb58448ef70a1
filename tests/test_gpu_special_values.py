"""Values at the end of the single-precision range: quaternions whose square overflows."""
import numpy as np
import pytest

from conftest import make_pair, per_env_error

pytestmark = pytest.mark.gpu
LARGEST = float(np.finfo(np.float32).max)


@pytest.mark.parametrize("index", [2, 3])
def test_a_quaternion_whose_square_overflows_turns_nothing(oracle_py, device, index):
    """The reciprocal root of an infinite square is zero: a base orientation of such a size, as a diverged environment has, turns
    into a zero quaternion, which the links below it read as none."""
    E = 16
    _, oracle, world, state = make_pair(oracle_py, device, index, E)
    state = {name: np.array(values) for name, values in state.items()}
    for env, size in ((3, 1.0e20), (5, 3.0e19), (9, LARGEST / 4.0)):
        state["base_pose"][env, 3:] *= np.float32(size)
    for w in (world, oracle):
        w.set_state(state)
        w.step()
    world.synchronize()
    assert np.array_equal(world.download("env_status"), oracle.download("env_status"))
    for name in ("link_pose", "articulation_qdd", "qdot"):
        got, expect = world.download(name), oracle.download(name)
        assert np.isfinite(expect).all() and np.isfinite(got).all(), name
        assert per_env_error(got, expect, E).max() <= 1e-4, name
    world.close()
    oracle.close()
