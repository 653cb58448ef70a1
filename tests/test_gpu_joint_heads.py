"""Joint rows' heads at the counts where the solve keeps them elsewhere: in their lanes' registers up to 64, as numbers beside
those up to 192, in the head fields past that."""
import numpy as np
import pytest

from conftest import nk, per_env_error
from test_gpu_head_capacity import crowded
from trees import tree_case

abi = nk.abi
pytestmark = pytest.mark.gpu
SOLVER_FAILURE = 1 << 13


@pytest.mark.parametrize("joints,limited,heads", [
    (20, 0, 20), (32, 16, 64), (33, 16, 65), (36, 36, 108), (44, 42, 128), (43, 43, 129), (60, 60, 180), (64, 64, 192)])
@pytest.mark.parametrize("contacts", [0, 2])
def test_joint_heads_match_the_oracle(oracle_py, device, joints, limited, heads, contacts):
    """Hinges on a fixed root, dry friction on every joint and both bounds of the first `limited` ones: a head each, beside
    two contact points or none."""
    E, most = 48, heads + contacts
    tree, desc, state = tree_case(oracle_py, joints, False, True, seed=joints, E=E, limb_joints=8, sphere_limbs=1 if contacts else 0)
    for l, link in enumerate(tree.template.links[1:]):
        link["frictionloss"] = 0.05 + 0.01 * (l % 5)
        if l < limited:
            link["lower"], link["upper"] = -0.3, 0.4
    world, oracle = nk.World(device, tree.template, desc), oracle_py.OracleWorld(tree.template, desc, threads=8)
    for w in (world, oracle):
        w.set_state(state)
        w.step()
    world.synchronize()
    rows = oracle.download("row_count")
    assert rows.max() == heads + 3 * contacts and np.array_equal(world.download("row_count"), rows), (rows.max(), most)
    assert not world.download("env_status").any() and not oracle.download("env_status").any()
    # single precision over as many heads, a step; the bar that the drives' tests hold
    for name in ("qdot", "q", "link_velocity"):
        error = per_env_error(world.download(name), oracle.download(name), E)
        assert error.max() <= 1e-4, (name, float(error.max()))


def test_contact_heads_past_the_capacity_leave_the_joint_heads_and_the_neighbours_alone(device):
    """240 contact points and 26 friction rows where 222 contacts fit: the environment is flagged, and no impulse lands outside
    the rows it has - the words past them, which belong to the next environment, hold what a world with fewer contacts has."""
    E = 3
    t, state = crowded(32, 240, 0.1, E, seed=32)
    up = dict(state, base_pose=state["base_pose"].copy())
    up["base_pose"][1, 2] += 5.0        # the second environment touches nothing
    world = nk.World(device, t, abi.world_desc(E, 1.0 / 240.0, vel_iters=8, contact_margin=0.1))
    world.set_state(up)
    world.step()
    world.synchronize()
    status = world.download("env_status")
    assert status[0] & SOLVER_FAILURE and status[2] & SOLVER_FAILURE and not status[1]
    assert np.all(np.isfinite(world.download("qdot")))
    alone = nk.World(device, t, abi.world_desc(1, 1.0 / 240.0, vel_iters=8, contact_margin=0.1))
    alone.set_state({k: v[1:2] for k, v in up.items()})
    alone.step()
    alone.synchronize()
    for name in ("lambda", "qdot", "link_velocity"):
        assert np.array_equal(world.download(name).reshape(E, -1)[1], alone.download(name).reshape(-1)), name
