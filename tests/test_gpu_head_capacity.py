"""Environments with as many live contact heads as a solve holds: its LDS takes a number of heads that falls with the
block's width, and what else a block keeps there must leave that number alone."""
import numpy as np
import pytest

from conftest import nk
from test_gpu_parity import ORACLE_OPS, bar, one_ulp_sensitivity, scaled_errors, velocity_scale
from trees import make_tree

pytestmark = pytest.mark.gpu
abi = nk.abi
SOLVER_FAILURE = 1 << 13
FLAT = (0.70710678, 0.70710678, 0.0, 0.0)      # a capsule lies along its own z


def crowded(dof, heads, friction, E, seed):
    """(template, state): a robot on a floating root whose underside is a field of capsules, two contact points each (and a
    sphere for an odd number), all of them in the plane's reach."""
    tree = make_tree(dof, True, True, seed, sphere_limbs=0)
    t = tree.template
    for l, link in enumerate(t.links):
        if friction and link["joint_type"] == abi.JOINT_REVOLUTE:
            link["frictionloss"] = friction
    g = np.random.default_rng(seed + 1)
    for k in range((heads + 1) // 2):
        at = (float(g.uniform(-0.3, 0.3)), float(g.uniform(-0.3, 0.3)), -0.1)
        if 2 * k + 1 < heads:
            t.add_body(abi.ROLE_PROXY, link=0, kind=abi.SHAPE_CAPSULE, params=(0.02, 0.02, 0, 0), local_pos=at, local_rot=FLAT, contype=1,
                       conaffinity=2, profile=0)
        else:
            t.add_body(abi.ROLE_PROXY, link=0, kind=abi.SHAPE_SPHERE, params=(0.02, 0, 0, 0), local_pos=at, contype=1, conaffinity=2, profile=0)
    nl = t.link_count
    q, qd, tau = (g.normal(0.0, s, (E, nl)).astype(np.float32) for s in (0.3, 0.5, 2.0))
    q[:, 0] = qd[:, 0] = tau[:, 0] = 0.0
    base = np.zeros((E, 7), np.float32)
    base[:, 2] = 0.12 - g.uniform(0.0, 0.002, E)
    base[:, 3] = 1.0
    return t, dict(q=q, qdot=qd, tau=tau, base_pose=base, root_twist=g.normal(0.0, 0.3, (E, 6)).astype(np.float32))


# (coordinates, joint friction, contact heads): what 150 KB of LDS hold of heads (a contact head 60 words and three rows of
# the block's width, a joint row's unit head 31) beside the block's two factors
CASES = [(12, 0.0, 393), (16, 0.0, 347), (20, 0.0, 310), (24, 0.0, 279), (28, 0.0, 253), (32, 0.0, 230), (20, 0.1, 303), (32, 0.1, 222),
         (36, 0.0, 218)]


@pytest.mark.parametrize("dof,friction,heads", CASES)
def test_a_solve_holds_the_heads_its_width_allows(oracle_py, device, dof, friction, heads):
    E = 4
    t, state = crowded(dof, heads, friction, E, seed=dof)
    # (sixteen sweeps bring every environment to the velocity tolerance; at a cap of eight some stop between two iterates
    # that differ by more than it, and a rounding decides how far: 1.2e-4 of the free velocity at 12 coordinates)
    desc = abi.world_desc(E, 1.0 / 240.0, vel_iters=64, contact_margin=0.1)
    sens = one_ulp_sensitivity(oracle_py, t, desc, state)
    world, oracle = nk.World(device, t, desc), oracle_py.OracleWorld(t, desc, threads=8)
    assert world.dof == dof
    for w in (world, oracle):
        w.set_state(state)
    for name, call in ORACLE_OPS.items():
        if name == "BlockDescentSolve":
            scale = velocity_scale(world, oracle, E)
        oracle.op(*call)
        world.op(name)
        if name == "BlockDescentSolve":
            break
    world.synchronize()
    assert np.array_equal(world.download("contact_count"), np.full(E, heads)) and np.array_equal(oracle.download("contact_count"), np.full(E, heads))
    assert not world.download("env_status").any() and not oracle.download("env_status").any()
    assert oracle.download("vbd_velocity_sweep_count").max() < 64
    error = scaled_errors(world.download("qdot_flat"), oracle.download("qdot_flat"), scale, E)
    print(f"dof {dof}, {heads} heads: velocities {error.max():.2e} from the oracle's, its own one-ulp sensitivity {sens['velocity']:.2e}")
    # two solves that meet the velocity tolerance (1e-5 m/s) may stop that far apart beside what a rounding moves them by
    assert np.all(error <= bar(sens, "velocity") + 1e-5 / scale)
    world.close()
    oracle.close()


def test_heads_past_the_capacity_flag_the_environment(device):
    E = 3
    t, state = crowded(32, 240, 0.0, E, seed=5)
    world = nk.World(device, t, abi.world_desc(E, 1.0 / 240.0, vel_iters=8, contact_margin=0.1))
    world.set_state(state)
    world.step()
    world.synchronize()
    assert np.all(world.download("env_status") & SOLVER_FAILURE)
    assert np.all(np.isfinite(world.download("qdot")))
    world.close()
