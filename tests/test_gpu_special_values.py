"""Values at the end of the single-precision range: quaternions whose square overflows, armatures that hold a joint."""
import numpy as np
import pytest

from conftest import make_pair, nk, per_env_error
from trees import tree_case

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


@pytest.mark.parametrize("armature", [1.0e30, LARGEST])
@pytest.mark.parametrize("from_last", [1, 9])
@pytest.mark.parametrize("rows", [False, True])
def test_a_joint_held_by_its_armature_leaves_the_others_moving(oracle_py, device, armature, from_last, rows):
    """Armatures are taken up to the largest float: a pivot whose reciprocal is no normal number, in the mass matrix's factor and
    beside dry friction on every joint."""
    E = 48
    tree, desc, state = tree_case(oracle_py, 20, False, True, seed=20, E=E, limb_joints=8, sphere_limbs=1)
    for l, link in enumerate(tree.template.links[1:]):
        link["frictionloss"] = 0.05 + 0.01 * (l % 5) if rows else 0.0
    tree.template.links[-from_last]["armature"] = armature
    world, oracle = nk.World(device, tree.template, desc), oracle_py.OracleWorld(tree.template, desc, threads=8)
    for w in (world, oracle):
        w.set_state(state)
        w.step()
    world.synchronize()
    assert not oracle.download("env_status").any() and not world.download("env_status").any()
    for name in ("articulation_qdd", "qdot", "link_velocity"):
        error = per_env_error(world.download(name), oracle.download(name), E)
        assert error.max() <= 1e-4, (name, float(error.max()))
    world.close()
    oracle.close()
