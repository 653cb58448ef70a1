"""An environment's solve and its rows are its own, whatever kernels and launches its batch takes: wide blocks two a SIMD, launches of as
many blocks as the machine holds, row assemblies of eight environments a wavefront."""
import numpy as np
import pytest

from conftest import nk
from trees import tree_case

abi = nk.abi
pytestmark = pytest.mark.gpu
SOLVER_FAILURE = 1 << 13
FIELDS = ("q", "qdot", "link_velocity", "lambda", "vbd_velocity_sweep_count", "env_status", "solver_residual")


def repeated(state, E):
    return {name: np.ascontiguousarray(np.asarray(v)[np.arange(E) % len(v)]) for name, v in state.items()}


def batches_agree(device, template, desc_of, state, small, large, steps=2, fields=FIELDS, failing=None, width=None, slots=False):
    """The environments of a large batch, the small one's over and over, step as the small one's do, bit for bit; those whose solve
    fails (`failing`, of the small batch) are flagged, and what becomes of them is nobody's concern."""
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
        kept = np.ones(small, bool) if failing is None else ~failing
        assert np.array_equal(b.view(np.uint8)[np.resize(kept, large)], a.view(np.uint8)[np.arange(large) % small][np.resize(kept, large)]), name
        if name == "env_status":
            assert np.array_equal((b[:, 0] & SOLVER_FAILURE) != 0, np.resize(~kept, large))
    assert width is None or many.info.solver_width == width
    blocks = few.info.solver_blocks_per_cu, many.info.solver_blocks_per_cu
    held = few.info.contact_slots_per_env
    few.close()
    many.close()
    return held if slots else blocks


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


def with_dry_friction(template):
    for link in template.links:
        if link["joint_type"] == abi.JOINT_REVOLUTE:
            link["frictionloss"] = 0.1
    return template


# Blocks with joint rows (general), blocks whose sweeps are narrower than their coordinates (reduced) and batches of 6144 on (dense) of over a third
# more environments than the machine holds blocks: the launches that have a queue.  The second number is the width of the sweeps.
@pytest.mark.parametrize("index,width,driven,large", [(2, 18, True, 2740), (2, 18, False, 6145), (3, 20, False, 2740), (3, 36, True, 2740)])
@pytest.mark.parametrize("sick", [False, True])
def test_environments_past_the_blocks_held_step_as_the_first(device, index, width, driven, large, sick):
    """Those that wait in the queue, one at the least; also behind environments whose velocity is no number, which leave their block's
    LDS to the next as the failed solve left it."""
    cfg = nk.synthetic.config(index, 150)
    template, state = with_dry_friction(cfg.template) if driven else cfg.template, cfg.state()
    failing = np.arange(150) % 4 == 1
    if sick:
        state["root_twist"] = np.where(failing[:, None], np.float32(np.nan), state["root_twist"]).astype(np.float32)
    blocks = batches_agree(device, template, lambda E: abi.world_desc(E, cfg.dt, vel_iters=cfg.vel_iters), state, 150, large, steps=1 if sick else 3,
                           failing=failing if sick else None, width=width)
    assert large > 256 * blocks[1] * 4 // 3   # (the queue's)


@pytest.mark.parametrize("dof,width,floating,limb_joints,sphere_limbs,driven,large", [
    (3, 3, False, 7, None, True, 2740), (7, 7, False, 3, None, True, 2740), (11, 11, True, 3, None, True, 2740), (14, 14, True, 3, None, True, 2740),
    (23, 23, True, 3, None, True, 2740), (26, 26, True, 3, None, True, 2740), (32, 32, True, 3, None, True, 2740),
    (24, 12, True, 3, 2, False, 2740), (27, 16, True, 3, 2, False, 2740), (32, 16, True, 5, 2, False, 2740), (40, 20, True, 7, 2, False, 2740),
    (44, 24, True, 7, 2, False, 2740), (48, 24, True, 7, 2, False, 2740), (51, 28, True, 7, 3, False, 2740), (56, 28, True, 7, 3, False, 2740),
    (60, 32, True, 7, 3, False, 2740), (64, 32, True, 7, 3, False, 2740), (24, 12, True, 3, 2, False, 6200), (8, 8, False, 3, None, False, 6200),
])
def test_trees_past_the_blocks_held_step_as_the_first(oracle_py, device, dof, width, floating, limb_joints, sphere_limbs, driven, large):
    """The same at the padded widths that the configurations leave out."""
    tree, _, state = tree_case(oracle_py, dof, floating, True, seed=7 * dof, E=48, limb_joints=limb_joints, sphere_limbs=sphere_limbs)
    template = with_dry_friction(tree.template) if driven else tree.template
    blocks = batches_agree(device, template, lambda E: abi.world_desc(E, 1.0 / 240.0, vel_iters=6), state, 48, large, width=width)
    assert large > 256 * blocks[1] * 4 // 3   # (the queue's)


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


ROW_FIELDS = ("lambda", "chain_jacobian", "chain_jacobian_b", "row_penetration", "row_cj_point", "row_cj_point_b", "row_cj_link", "ucontact_count", "row_count",
              "contact_material", "env_status", "qdot_flat", "q", "qdot", "link_velocity", "contact_row_extent")


@pytest.mark.parametrize("dof,floating,branched,limb_joints,sphere_pairs", [
    (8, False, True, 2, False), (7, True, False, 7, False), (6, False, False, 7, False), (2, False, False, 2, False), (4, False, True, 2, True), (8, True, True, 1, True),
])
def test_trees_whose_rows_are_assembled_eight_a_wavefront_step_as_alone(oracle_py, device, dof, floating, branched, limb_joints, sphere_pairs):
    """One point a slot, up to eight slots; spheres of different limbs too, whose rows have the articulation on both sides."""
    small = 70
    tree, _, state = tree_case(oracle_py, dof, floating, branched, seed=11 * dof, E=small, limb_joints=limb_joints, sphere_pairs=sphere_pairs)
    slots = batches_agree(device, tree.template, lambda E: abi.world_desc(E, 1.0 / 240.0, vel_iters=6, contact_margin=0.1), state, small, 2051, steps=3, fields=ROW_FIELDS,
                          slots=True)
    assert 1 <= slots <= 8


def test_two_boxes_on_a_tree_whose_rows_are_assembled_eight_a_wavefront_step_as_alone(device):
    """Two slots of four points each, a root and the link on its hinge: every lane a place."""
    small, g = 70, np.random.default_rng(3)
    t = abi.Template()
    t.add_link(abi.JOINT_FLOATING, None, mass=3.0, diag_inertia=(0.03, 0.04, 0.05))
    t.add_link(abi.JOINT_REVOLUTE, 0, axis=(0, 1, 0), local_pos=(0.35, 0, 0), mass=1.0, diag_inertia=(0.01, 0.01, 0.01), armature=0.02)
    profile = t.add_profile(0.6)
    t.add_body(abi.ROLE_STATIC, kind=abi.SHAPE_PLANE, contype=2, conaffinity=1, profile=profile)
    for link, half in ((0, (0.15, 0.1, 0.1)), (1, (0.1, 0.1, 0.1))):
        t.add_body(abi.ROLE_LINK_BODY, link=link, kind=abi.SHAPE_NONE, contype=0, conaffinity=0)
        t.add_body(abi.ROLE_PROXY, link=link, kind=abi.SHAPE_BOX, params=(*half, 0), contype=1, conaffinity=2, profile=profile)
    t.max_contacts_per_env = 2
    base = np.zeros((small, 7), np.float32)
    base[:, 2] = 0.1 + g.uniform(-0.004, 0.02, small)
    base[:, 3] = 1.0
    base[:, 4:] = 0.5 * g.normal(0.0, 0.02, (small, 3))
    base[:, 3:] /= np.linalg.norm(base[:, 3:], axis=1, keepdims=True)
    state = dict(q=np.stack([np.zeros(small), g.normal(0.0, 0.05, small)], 1).astype(np.float32), qdot=np.zeros((small, 2), np.float32), tau=np.zeros((small, 2), np.float32),
                 base_pose=base, root_twist=g.normal(0.0, 0.3, (small, 6)).astype(np.float32))
    slots = batches_agree(device, t, lambda E: abi.world_desc(E, 1.0 / 240.0, vel_iters=8, contact_margin=0.02), state, small, 2051, steps=4, fields=ROW_FIELDS, slots=True)
    assert slots == 2
