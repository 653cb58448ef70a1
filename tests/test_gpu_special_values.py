"""Values at the end of the single-precision range: quaternions whose square overflows, armatures that hold a joint, impulses
whose size is a subnormal number."""
import numpy as np
import pytest

from conftest import make_pair, nk, per_env_error
from test_gpu_parity import UPSTREAM, both
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


@pytest.mark.parametrize("size", [1.0e-36, 3.0e-38, 2.0e-39, 1.0e-40, 1.0e-42])
@pytest.mark.parametrize("index,driven", [(2, False), (3, False), (2, True)])
def test_a_tangential_impulse_of_any_size_has_a_direction_on_the_elliptic_cone(oracle_py, device, index, driven, size):
    """Contacts without a normal impulse whose tangents ask for one of `size`: on the cone, whose direction is the quotient of the
    tangents by their length, also where that is too small to have a reciprocal.  At the full width, reduced and beside joint rows."""
    E = 8
    cfg = nk.synthetic.config(index, E)
    for profile in cfg.template.profiles:
        profile["law"] = nk.abi.LAW_MUJOCO
    cfg.template.contact_cone = nk.abi.CONE_ELLIPTIC
    if driven:
        for link in cfg.template.links[1:]:
            link["frictionloss"] = 0.1
    desc = nk.abi.world_desc(E, cfg.dt, vel_iters=cfg.vel_iters)
    world, oracle = nk.World(device, cfg.template, desc), oracle_py.OracleWorld(cfg.template, desc, threads=8)
    state = cfg.state()
    for w in (world, oracle):
        w.set_state(state)
    for name in UPSTREAM:
        both(oracle, world, name)
    R = world.rows_per_env
    rows = oracle.download("urows").reshape(E, R, -1).copy()
    tangent = rows[:, :, 0].copy().view(np.uint32) & 0b1001 == 0b1001   # active block tangents
    g = np.random.default_rng(index)
    rows[:, :, 4] = np.where(tangent, g.choice([-1.0, 1.0], (E, R)) * g.uniform(0.3, 1.0, (E, R)) * size / cfg.dt, 0.0)
    assert tangent.any(1).sum() >= E // 2
    for w in (world, oracle):
        w.upload("urows", rows)
        for name in ("qdot", "link_velocity"):
            w.upload(name, np.zeros_like(w.download(name)))
    both(oracle, world, "BlockDescentSolve")
    assert not oracle.download("env_status").any() and not world.download("env_status").any()
    got, expect = world.download("lambda").reshape(E, R), oracle.download("lambda").reshape(E, R)
    assert (expect[tangent] != 0.0).all() and np.isfinite(got).all()
    # a word of the quotients and products on the way carries the spacing of the subnormal numbers, 2^-149, beside a rounding
    assert np.abs(got - expect).max() <= 1e-5 * np.abs(expect).max() + 64 * 2.0 ** -149
    assert np.abs(world.download("qdot")).max() <= 1e-6 and np.abs(world.download("link_velocity")).max() <= 1e-6
    world.close()
    oracle.close()
