"""A step's result is the environment's own, whatever kernels and launches its batch takes: wide blocks two a SIMD, launches of as
many blocks as the machine holds, row assemblies of eight environments a wavefront."""
import numpy as np
import pytest

from conftest import nk
from trees import tree_case

abi = nk.abi
pytestmark = pytest.mark.gpu
FIELDS = ("q", "qdot", "link_velocity", "lambda", "vbd_velocity_sweep_count", "env_status", "solver_residual")


def repeated(state, E):
    return {name: np.ascontiguousarray(np.asarray(v)[np.arange(E) % len(v)]) for name, v in state.items()}


def batches_agree(device, template, desc_of, state, small, large, steps=2, fields=FIELDS):
    """The environments of a large batch, the small one's over and over, step as the small one's do, bit for bit."""
    few, many = nk.World(device, template, desc_of(small)), nk.World(device, template, desc_of(large))
    few.set_state(state)
    many.set_state(repeated(state, large))
    for _ in range(steps):
        few.step()
        many.step()
    few.synchronize()
    many.synchronize()
    assert (few.download("contact_count") > 0).any()
    for name in fields:
        a, b = few.download(name).reshape(small, -1), many.download(name).reshape(large, -1)
        assert np.array_equal(b.view(np.uint8), a.view(np.uint8)[np.arange(large) % small]), name
    blocks = few.info.solver_blocks_per_cu, many.info.solver_blocks_per_cu
    few.close()
    many.close()
    return blocks


@pytest.mark.parametrize("dof,floating,branched,limb_joints", [
    (37, False, True, 2), (40, False, False, 7), (44, True, True, 3), (50, True, True, 2), (53, False, True, 4), (57, True, False, 7),
    (61, False, True, 2), (64, False, True, 3),
])
def test_wide_trees_two_a_simd_step_as_one_a_simd(oracle_py, device, dof, floating, branched, limb_joints):
    """Every padded width, with coordinates that fill it and that do not, ways and heads that are runs of lanes and that are not."""
    small, large = 48, 3329   # (fewer heads than coordinates: paired from 3328 environments on)
    tree, _, state = tree_case(oracle_py, dof, floating, branched, seed=5 * dof, E=small, limb_joints=limb_joints)
    blocks = batches_agree(device, tree.template, lambda E: abi.world_desc(E, 1.0 / 240.0, vel_iters=6), state, small, large)
    assert blocks[0] <= 4 < blocks[1]


@pytest.mark.parametrize("dof,large", [(40, 3328), (44, 3333), (64, 3329), (64, 3327)])
def test_a_wide_blocks_mass_factor_takes_the_packed_rows_room(oracle_py, device, dof, large):
    """n (n + 1) / 2 words of the padded width, a multiple of four: what a caller that binds its own memory gives for it, whichever
    build solves.  The paired build's words past its factor stay as they are."""
    tree, _, state = tree_case(oracle_py, dof, True, True, seed=5 * dof, E=48, limb_joints=3)
    w = nk.World(device, tree.template, abi.world_desc(large, 1.0 / 240.0, vel_iters=2))
    room = (dof * (dof + 1) // 2 + 3) // 4 * 4
    assert w.download("solver_mass_factor").size == large * room
    assert (w.info.solver_blocks_per_cu > 4) == (large >= 3328)
    words = np.full((large, room), 7.0, np.float32)
    w.upload("solver_mass_factor", words)
    w.set_state(repeated(state, large))
    w.step()
    w.synchronize()
    words = w.download("solver_mass_factor").reshape(large, room)
    if large >= 3328:   # 8 quads^2 words by fours, four zeros, a word a quad
        quads = dof // 4
        used = 8 * quads * quads + 4 + quads
        assert (words[:, used:] == 7.0).all() and not (words[:, :used] == 7.0).any()
        assert not words[:, 8 * quads * quads:8 * quads * quads + 4].any()
    w.close()


@pytest.mark.parametrize("large,held", [(2111, 8), (2047, 4)])
def test_ropes_two_a_simd_step_as_one_a_simd(device, large, held):
    """As many heads as coordinates: paired from 2048 environments on."""
    cfg = nk.synthetic.config(5, 64)
    blocks = batches_agree(device, cfg.template, lambda E: abi.world_desc(E, cfg.dt, vel_iters=cfg.vel_iters), cfg.state(), 64, large)
    assert blocks == (4, held)


@pytest.mark.parametrize("index,driven,large", [(2, False, 2049), (2, False, 6144 + 1), (3, False, 2600), (3, True, 1900)])
def test_environments_past_the_blocks_held_step_as_the_first(device, index, driven, large):
    """Two-wave, dense and general kernels with more environments than blocks: the ones that wait in the queue, one at the least."""
    cfg = nk.synthetic.config(index, 150)
    template = cfg.template
    if driven:
        for link in template.links:
            if link["joint_type"] == abi.JOINT_REVOLUTE:
                link["frictionloss"] = 0.1
    batches_agree(device, template, lambda E: abi.world_desc(E, cfg.dt, vel_iters=cfg.vel_iters), cfg.state(), 150, large, steps=3)


@pytest.mark.parametrize("large", [2048, 2051])
def test_boxes_whose_rows_are_assembled_eight_a_wavefront_step_as_alone(device, large):
    """Four-point manifolds that come and go: some environments have no point, some a few."""
    cfg = nk.synthetic.config(6, 70)
    state = cfg.state()
    state["base_pose"] = state["base_pose"].copy()
    state["base_pose"][::3, 2] += np.linspace(0.0, 0.03, len(state["base_pose"][::3]), dtype=np.float32)
    state["base_pose"][1::5, 4] += 0.08
    state["base_pose"][:, 3:] /= np.linalg.norm(state["base_pose"][:, 3:], axis=1, keepdims=True)
    batches_agree(device, cfg.template, lambda E: abi.world_desc(E, cfg.dt, vel_iters=cfg.vel_iters), state, 70, large, steps=4,
                  fields=("lambda", "chain_jacobian", "chain_jacobian_b", "row_penetration", "row_cj_point", "ucontact_count", "row_count",
                          "contact_material", "body_linear_velocity", "body_angular_velocity", "base_pose", "env_status", "qdot_flat"))
