"""Reduced blocks under the elliptic cone of the MuJoCo law at every compiled pair of widths, against the oracle, which
solves the full block; full blocks under it, and blocks of many heads."""
import numpy as np
import pytest

from conftest import nk
from test_gpu_head_capacity import crowded
from test_gpu_parity import ORACLE_OPS, UPSTREAM, bar, close, one_ulp_sensitivity, scaled_errors, velocity_scale
from test_gpu_widths import REDUCED
from trees import tree_case

pytestmark = pytest.mark.gpu
abi = nk.abi


@pytest.mark.parametrize("pairs", [False, True])
@pytest.mark.parametrize("dof,floating,limb_joints,sphere_limbs,width", REDUCED)
def test_elliptic_reduced_blocks_match_the_oracle(oracle_py, device, dof, floating, limb_joints, sphere_limbs, width, pairs):
    E = 40
    tree, desc, state = tree_case(oracle_py, dof, floating, True, seed=5 * dof + sphere_limbs, E=E, limb_joints=limb_joints,
                                  sphere_limbs=sphere_limbs, sphere_pairs=pairs)
    for profile in tree.template.profiles:
        profile["law"] = abi.LAW_MUJOCO
    tree.template.contact_cone = abi.CONE_ELLIPTIC
    oracle = oracle_py.OracleWorld(tree.template, desc, threads=8)
    world = nk.World(device, tree.template, desc)
    assert world.info.solver_width == width
    oracle.set_state(state)
    world.set_state(state)
    sens = one_ulp_sensitivity(oracle_py, tree.template, desc, state)
    oracle.step()
    world.step()
    world.synchronize()
    assert not world.download("env_status").any() and not oracle.download("env_status").any()
    assert (oracle.download("contact_count") > 0).mean() >= 0.4
    for name in ("qdot_flat", "link_velocity"):   # the eliminated coordinates among them
        close(world, oracle, name, tol=bar(sens, "velocity"))
    world.close()
    oracle.close()


@pytest.mark.parametrize("dof,floating", [(4, False), (7, False), (8, True), (12, True), (16, False), (18, True), (20, True), (21, True)])
def test_elliptic_full_blocks_match_the_oracle(oracle_py, device, dof, floating):
    """Contact heads alone under the cone at the full width: kernels of their own up to 20 coordinates, the general one past them."""
    E = 40
    tree, desc, state = tree_case(oracle_py, dof, floating, False, seed=7 * dof, E=E)
    for profile in tree.template.profiles:
        profile["law"] = abi.LAW_MUJOCO
    tree.template.contact_cone = abi.CONE_ELLIPTIC
    oracle = oracle_py.OracleWorld(tree.template, desc, threads=8)
    world = nk.World(device, tree.template, desc)
    assert world.info.solver_width == dof
    oracle.set_state(state)
    world.set_state(state)
    sens = one_ulp_sensitivity(oracle_py, tree.template, desc, state)
    oracle.step()
    world.step()
    world.synchronize()
    assert not world.download("env_status").any() and not oracle.download("env_status").any()
    assert (oracle.download("contact_count") > 0).any()
    close(world, oracle, "qdot_flat", tol=bar(sens, "velocity"))
    world.close()
    oracle.close()


# (coordinates, heads, joint friction, width of the sweeps): the line search takes up to sixteen heads in a row of lanes, up to 64 a
# lane each, and reads the ones past that as it goes; a world of more than 64, or with joint rows, takes the general kernel
@pytest.mark.parametrize("dof,heads,friction,width", [(8, 16, 0.0, 8), (8, 17, 0.0, 8), (12, 40, 0.0, 12), (20, 33, 0.0, 20), (20, 64, 0.0, 20),
                                                      (24, 17, 0.0, 12), (36, 40, 0.0, 20), (64, 64, 0.0, 32), (20, 66, 0.0, 20), (24, 100, 0.0, 24),
                                                      (12, 15, 0.1, 12), (20, 40, 0.1, 20)])
def test_many_elliptic_heads_match_the_oracle(oracle_py, device, dof, heads, friction, width):
    E = 8
    t, state = crowded(dof, heads, friction, E, seed=dof + heads)
    for profile in t.profiles:
        profile["law"] = abi.LAW_MUJOCO
    t.contact_cone = abi.CONE_ELLIPTIC
    desc = abi.world_desc(E, 1.0 / 240.0, vel_iters=64, contact_margin=0.1)
    sens = one_ulp_sensitivity(oracle_py, t, desc, state)
    world, oracle = nk.World(device, t, desc), oracle_py.OracleWorld(t, desc, threads=8)
    assert world.dof == dof and world.info.solver_width == width
    for w in (world, oracle):
        w.set_state(state)
    for name in UPSTREAM:
        oracle.op(*ORACLE_OPS[name])
        world.op(name)
    scale = velocity_scale(world, oracle, E)
    oracle.op(*ORACLE_OPS["BlockDescentSolve"])
    world.op("BlockDescentSolve")
    world.synchronize()
    R = world.rows_per_env
    flags = oracle.download("urows").reshape(E, R, -1)[:, :, 0].copy().view(np.uint32)
    live = ((flags & 1 != 0) & (flags & (1 << 3) == 0) & (flags & (1 << 2) != 0)).sum(1)   # three axes each
    assert (live == heads).all(), live
    assert not world.download("env_status").any() and not oracle.download("env_status").any()
    error = scaled_errors(world.download("qdot_flat"), oracle.download("qdot_flat"), scale, E)
    print(f"dof {dof}, {heads} heads: velocities {error.max():.2e} from the oracle's, its own one-ulp sensitivity {sens['velocity']:.2e}")
    # two solves that meet the velocity tolerance (1e-5 m/s) may stop that far apart beside what a rounding moves them by
    assert oracle.download("vbd_velocity_sweep_count").max() < 64
    assert np.all(error <= bar(sens, "velocity") + 1e-5 / scale)
    world.close()
    oracle.close()
