"""Wide blocks sum over heads and coordinates as differences of running sums where those are neighbours for every coordinate
or head, and over each lane's own choice elsewhere."""
import numpy as np
import pytest

from conftest import nk
from test_gpu_parity import bar, close, compare_ops, one_ulp_sensitivity
from trees import tree_case

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dof,floating,branched,limb_joints", [
    (38, False, False, 7),    # a chain: heads and coordinates are runs, of lanes that a row of sixteen ends in
    (64, False, False, 7),    # up to the last lane
    (46, True, False, 7),     # a chain on a floating root: its six coordinates head every way
    (46, True, True, 2),      # limbs in turn: the heads are runs, the ways are not
])
@pytest.mark.parametrize("order", ["as they come", "apart"])
def test_heads_in_any_order_match_the_oracle(oracle_py, device, dof, floating, branched, limb_joints, order):
    """The order of the spheres' rows is that of the contact heads: with every second one first, a limb's heads are no
    neighbours."""
    E = 32
    tree, desc, state = tree_case(oracle_py, dof, floating, branched, seed=17 * dof + branched, E=E, limb_joints=limb_joints)
    heads = len(tree.sphere_links)
    if order == "apart":
        spheres = tree.template.bodies[-heads:]
        tree.template.bodies[-heads:] = spheres[1::2] + spheres[0::2]
    oracle, world = oracle_py.OracleWorld(tree.template, desc, threads=8), nk.World(device, tree.template, desc)
    assert world.dof == dof
    for w in (oracle, world):
        w.set_state(state)
    sens = one_ulp_sensitivity(oracle_py, tree.template, desc, state)
    compare_ops(oracle, world, E, sens, state)
    assert (oracle.download("contact_count") > 0).mean() >= 0.4
    close(world, oracle, "link_velocity", tol=bar(sens, "velocity"))
    world.close()
    oracle.close()
