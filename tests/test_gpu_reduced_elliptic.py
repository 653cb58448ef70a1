"""Reduced blocks under the elliptic cone of the MuJoCo law at every compiled pair of widths, against the oracle, which
solves the full block."""
import pytest

from conftest import nk
from test_gpu_parity import bar, close, one_ulp_sensitivity
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
