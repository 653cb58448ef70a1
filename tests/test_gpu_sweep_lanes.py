"""The tree sweeps (world poses, link twists) give an environment a share of a wavefront's lanes that depends on its links
and on the number of environments: each share, at the edges where it begins and ends, against the share of a small batch,
which the other tests hold to the oracle.  The lanes of an environment run the same device code whatever their number, so
the outputs are the same bit for bit."""
import numpy as np
import pytest

from conftest import nk
from test_gpu_parity import close

abi = nk.abi
pytestmark = pytest.mark.gpu


def chain(links, floating):
    """`links` links in two chains below the root; the joints from the 60th on are fixed ones, so that there are no more
    coordinates than a block holds."""
    t = abi.Template()
    t.add_link(abi.JOINT_FLOATING if floating else abi.JOINT_FIXED, None, mass=2.0, diag_inertia=(0.05, 0.06, 0.07))
    for l in range(1, links):
        kind = (abi.JOINT_REVOLUTE, abi.JOINT_REVOLUTE, abi.JOINT_PRISMATIC)[l % 3] if l < 55 else abi.JOINT_FIXED
        t.add_link(kind, max(l - 2, 0), axis=((1, 0, 0), (0, 1, 0), (0, 0, 1))[l % 3], local_pos=(0.02 * (l % 2), 0.01, -0.05), mass=0.3,
                   diag_inertia=(0.002, 0.003, 0.004), com=(0.0, 0.0, -0.02), armature=0.02)
    return t


def seeded(links, envs, floating, seed):
    g = np.random.default_rng(seed)
    normal = lambda s, *shape: (s * g.standard_normal(shape)).astype(np.float32)   # noqa: E731
    state = dict(q=normal(0.2, envs, links), qdot=normal(0.3, envs, links), tau=normal(0.2, envs, links),
                 base_pose=np.zeros((envs, 7), np.float32), root_twist=normal(0.3, envs, 6) * np.float32(floating))
    for name in ("q", "qdot", "tau"):
        state[name][:, 0] = 0.0
    state["base_pose"][:, 3] = 1.0
    if floating:
        state["base_pose"][:, :3] = normal(0.5, envs, 3)
        state["base_pose"][:, 4:] = normal(0.1, envs, 3)
        state["base_pose"][:, 3:] /= np.linalg.norm(state["base_pose"][:, 3:], axis=1, keepdims=True)
    return state


CASES = [  # links, environments: 8 lanes from 8192 environments on, 16 from 4096, 32 from 2048; 64; two links a lane; more than two
    (1, 8193), (7, 8197), (8, 8192), (8, 8191), (9, 8195), (16, 4096), (16, 4099), (16, 4095), (17, 4097), (31, 2049), (32, 2048), (32, 2047),
    (33, 2049), (64, 2049), (65, 67), (128, 65), (130, 67),
]


@pytest.mark.parametrize("graph", [False, True])
@pytest.mark.parametrize("links,envs", CASES)
def test_every_share_of_lanes_gives_the_bits_of_a_small_batch(oracle_py, device, links, envs, graph):
    floating = links % 2 == 1
    t, few = chain(links, floating), 16
    state = seeded(links, envs, floating, links + envs)
    ends = np.r_[0:few // 2, envs - few // 2:envs]                   # the first and the last environments: the last wavefront is part full
    part = {name: np.ascontiguousarray(value[ends]) for name, value in state.items()}
    large, small = nk.World(device, t, abi.world_desc(envs, 0.004)), nk.World(device, t, abi.world_desc(few, 0.004))
    oracle = oracle_py.OracleWorld(t, abi.world_desc(few, 0.004), threads=4)
    for world, values in ((large, state), (small, part), (oracle, part)):
        world.set_state(values)
    for world in (large, small):
        world.op("FkWorldPoses"); world.op("FkLinkVelocities")       # the two sweeps as kernels of their own
        world.synchronize()
    for name in ("link_pose", "link_velocity"):
        assert np.array_equal(large.download(name).reshape(envs, -1)[ends], small.download(name).reshape(few, -1)), name
    for world in (large, small):
        world.set_execution_mode(graph)
        world.step(2)                                                # and behind the positions' integration in one
        world.synchronize()
    oracle.step(); oracle.step()
    for name in ("link_pose", "link_velocity", "q", "qdot", "base_pose"):
        assert np.array_equal(large.download(name).reshape(envs, -1)[ends], small.download(name).reshape(few, -1)), name
    close(small, oracle, "link_pose", tol=2e-4)                      # twice the bar of a step
    for world in (large, small, oracle):
        world.close()
