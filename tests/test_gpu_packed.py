"""The solve of small blocks four environments a wavefront (batches from 8192 on): the batch's edges, more heads than a pass
takes, articulated blocks and single-axis heads, against the kernel that gives an environment a wavefront and against the
oracle; and environments whose solve fails beside healthy ones."""
import numpy as np
import pytest

from conftest import nk, per_env_error
from rigid import body_field, box_template
from test_gpu_head_capacity import crowded
from test_gpu_parity import ORACLE_OPS, UPSTREAM, bar, one_ulp_sensitivity, scaled_errors, velocity_scale
from test_gpu_rigid import seeded_boxes
from trees import tree_case

pytestmark = pytest.mark.gpu
abi = nk.abi
STATE = ("qdot", "link_velocity", "lambda")


def repeated(values, count):
    values = np.asarray(values)
    return np.concatenate([values] * (count // len(values) + 1))[:count]


def copies_alike(big, name, E, count):
    """The batch repeats E environments: every copy holds the first one's bits."""
    batch = big.download(name).reshape(count, -1)
    assert np.array_equal(batch, repeated(batch[:E], count)), name
    return batch[:E]


# a last wavefront of one, two and three environments, and batches with and without environments that go alone; under the
# pyramidal cone the last batch that does not go four a wavefront and the first ones that do
@pytest.mark.parametrize("count", [8193, 8194, 8195, 12287, 12288, 12289, 12290, 12291, 24576, 24577])
@pytest.mark.parametrize("law", ["native", "pyramidal"])
def test_free_boxes_four_a_wavefront(device, count, law):
    E = 60
    t = box_template(half=(0.2, 0.15, 0.1), mass=3.0, diag=(0.03, 0.04, 0.05), mu=0.6)
    if law == "pyramidal":   # sixteen heads, on one axis each
        for profile in t.profiles:
            profile["law"] = abi.LAW_MUJOCO
        t.contact_cone = abi.CONE_PYRAMIDAL
    pose, v, w = seeded_boxes(E, 21)
    after = {}
    for envs in (E, count):
        world = nk.World(device, t, abi.world_desc(envs, 1.0 / 240.0, vel_iters=8, pos_iters=4, contact_margin=0.02))
        world.upload("base_pose", repeated(pose, envs))
        world.upload("body_linear_velocity", repeated(body_field(t, v), envs))
        world.upload("body_angular_velocity", repeated(body_field(t, w), envs))
        world.step(3); world.synchronize()
        names = ("base_pose", "body_linear_velocity", "body_angular_velocity", "lambda", "env_status", "vbd_velocity_sweep_count")
        after[envs] = {name: copies_alike(world, name, E, envs) for name in names}
        assert (world.download("contact_count") > 0).mean() >= 0.4
        world.close()
    for name, value in after[E].items():
        if law == "native" or value.dtype != np.float32:   # four heads, none of these states groups their sums otherwise: the same bits
            assert np.array_equal(value, after[count][name]), name
        else:   # the same sums in another grouping; three steps
            assert per_env_error(value, after[count][name], E, floor=1e-2).max() <= 3e-4, name


@pytest.mark.parametrize("dof,floating", [(4, False), (7, False), (8, True)])
def test_small_trees_four_a_wavefront(oracle_py, device, dof, floating):
    E, count = 48, 8192 + 31
    tree, desc, state = tree_case(oracle_py, dof, floating, True, seed=5 * dof + 1, E=E)
    small = nk.World(device, tree.template, desc)
    small.set_state(state)
    big = nk.World(device, tree.template, abi.world_desc(count, 1.0 / 240.0, vel_iters=8, contact_margin=0.1))
    big.set_state({k: repeated(v, count) for k, v in state.items()})
    for world in (small, big):
        assert world.dof == dof
        world.step(); world.synchronize()
    assert (small.download("contact_count") > 0).mean() >= 0.4, "the case must exercise the contact solve"
    sens = one_ulp_sensitivity(oracle_py, tree.template, desc, state)
    assert np.array_equal(copies_alike(big, "env_status", E, count).ravel(), small.download("env_status").ravel())
    for name in STATE:
        error = per_env_error(copies_alike(big, name, E, count), small.download(name), E).max()
        assert error <= bar(sens, "lambda" if name == "lambda" else "velocity"), (name, error)
    small.close(); big.close()


@pytest.mark.parametrize("count,packed", [(8192, False), (12287, False), (12288, True)])
def test_boxes_under_the_pyramidal_cone_go_four_a_wavefront_in_larger_batches(device, count, packed):
    """Six of the wavefronts of four fit a compute unit; they pay from 12288 environments on."""
    t = box_template(half=(0.2, 0.15, 0.1), mass=3.0, diag=(0.03, 0.04, 0.05), mu=0.6)
    for profile in t.profiles:
        profile["law"] = abi.LAW_MUJOCO
    t.contact_cone = abi.CONE_PYRAMIDAL
    world = nk.World(device, t, abi.world_desc(count, 1.0 / 240.0, vel_iters=8, contact_margin=0.02))
    assert (world.info.solver_blocks_per_cu == 6) == packed
    world.close()


def crowded_case(dof, heads, E):
    """A body of `dof` coordinates on `heads` contact points of three axes each, some of them in the air: tilted, at heights of
    their own."""
    t, state = crowded(dof, heads, 0.0, E, seed=10 * dof + heads)
    g = np.random.default_rng(heads)
    state["base_pose"][:, 2] = 0.12 + g.uniform(-0.003, 0.003, E)
    state["base_pose"][:, 4:] = 0.5 * g.normal(0.0, 0.02, (E, 3))
    state["base_pose"][:, 3:] /= np.linalg.norm(state["base_pose"][:, 3:], axis=1, keepdims=True)
    return t, state


# heads: a second pass of one and of four, a third of one, all sixteen (a wavefront's LDS lets ten, nine and six share a unit)
@pytest.mark.parametrize("dof,heads,blocks", [(8, 5, None), (7, 8, 10), (8, 9, 9), (8, 16, 6), (7, 15, 6)])
def test_blocks_of_many_three_axis_heads_match_the_oracle(oracle_py, device, dof, heads, blocks):
    """Velocities, impulses and the position pass's push-out, op by op, against the oracle in single and in double precision."""
    E, count = 48, 8192 + 48
    t, state = crowded_case(dof, heads, E)
    kw = dict(vel_iters=64, pos_iters=4, contact_margin=0.1)
    desc = abi.world_desc(E, 1.0 / 240.0, **kw)
    sens = one_ulp_sensitivity(oracle_py, t, desc, state)
    single, double = oracle_py.OracleWorld(t, desc, threads=8), oracle_py.OracleWorld(t, desc, threads=8, double=True)
    small = nk.World(device, t, desc)
    big = nk.World(device, t, abi.world_desc(count, 1.0 / 240.0, **kw))
    assert big.dof == dof and (blocks is None or big.info.solver_blocks_per_cu == blocks)
    for w in (single, double, small):
        w.set_state(state)
    big.set_state({k: repeated(v, count) for k, v in state.items()})
    for name in UPSTREAM + ["BlockDescentSolve"]:
        if name == "BlockDescentSolve":
            scale = velocity_scale(small, single, E)
        for w in (single, double):
            w.op(*ORACLE_OPS[name])
        for w in (small, big):
            w.op(name)
    big.synchronize()
    rows = single.download("urows").reshape(E, big.rows_per_env, -1)
    live = ((rows[:, :, 0].copy().view(np.uint32) & 0b1001) == 1).sum(1)   # active and no block's tangent
    pushed = (single.download("lambda").reshape(E, big.rows_per_env) != 0.0)
    assert (live > 4).mean() > 0.5 and live.max() == heads and (pushed.sum(1) > 4).any()
    assert not single.download("env_status").any() and not copies_alike(big, "env_status", E, count).any()
    got, expect = copies_alike(big, "qdot_flat", E, count), single.download("qdot_flat")
    allowed = bar(sens, "velocity") + 1e-5 / scale   # two solves that meet the velocity tolerance may stop that far apart
    assert (scaled_errors(got, expect, scale, E) <= allowed).all(), scaled_errors(got, expect, scale, E).max()
    assert (scaled_errors(got, small.download("qdot_flat"), scale, E) <= allowed).all()
    exact = double.download("qdot_flat")
    error, oracle_error = (scaled_errors(v, exact, scale, E) for v in (got, expect))
    print(f"dof {dof}, {heads} heads: from the double solve {error.max():.1e} (median {np.median(error):.1e}), "
          f"the oracle {oracle_error.max():.1e} (median {np.median(oracle_error):.1e})")
    assert np.median(error) <= max(2.0 * np.median(oracle_error), 1e-6)
    pushes = {name: copies_alike(big, name, E, count) for name in ("qdot_pseudo", "link_velocity_pseudo")}
    assert max(np.abs(v).max() for v in pushes.values()) > 1e-2, "the position pass must push"
    for name, value in pushes.items():   # one solve more, from the same rows
        size = np.abs(single.download(name)).reshape(E, -1).max(1) + 1e-2
        assert (scaled_errors(value, single.download(name), size, E) <= allowed + 1e-4).all(), name
    for w in (single, double, small, big):
        w.close()


SICK = ("velocity", "mass", "heads")


@pytest.mark.parametrize("case", ["box", "tree"])
def test_environments_whose_solve_fails_leave_the_others_of_their_wavefront_alone(device, case):
    """Every fifth environment of the batch has a velocity that is no number, a mass matrix with a negative pivot or more heads than
    its world holds: it is flagged, and the others end with the bits they end with beside healthy ones."""
    E = count = 8192 + 3
    kw = dict(vel_iters=8, pos_iters=4, contact_margin=0.05)
    if case == "box":
        t = box_template(half=(0.2, 0.15, 0.1), mass=3.0, diag=(0.03, 0.04, 0.05), mu=0.6)
        pose, v, w = seeded_boxes(E, 3)
    else:
        t, state = crowded_case(8, 6, E)
    after = {}
    for sick in (False, True):
        world = nk.World(device, t, abi.world_desc(count, 1.0 / 240.0, **kw))
        if case == "box":
            for name, values in (("base_pose", pose), ("body_linear_velocity", body_field(t, v)), ("body_angular_velocity", body_field(t, w))):
                world.upload(name, values)
        else:
            world.set_state(state)
        for name in (["IntegrateVelocity"] + UPSTREAM[:1] + UPSTREAM[2:] if case == "box" else UPSTREAM):   # a free body's dynamics
            world.op(name)
        world.synchronize()
        chosen = np.arange(0, count, 5)
        kind = (chosen // 5) % len(SICK)
        R, dof = world.rows_per_env, world.dof
        if sick:
            velocity = world.download("link_velocity").reshape(count, -1)
            velocity[chosen[kind == 0]] = np.nan
            world.upload("link_velocity", velocity)
            mass = world.download("m").reshape(count, -1)
            mass[chosen[kind == 1], 0] *= -1.0
            world.upload("m", mass)
            rows = world.download("urows").reshape(count, R, -1)
            flags = rows[:, :, 0].view(np.uint32)
            crowd = chosen[kind == 2]
            flags[crowd] &= ~np.uint32(1 << 3)   # the tangents stand as heads of their own
            world.upload("urows", rows)
        world.op("BlockDescentSolve")
        world.synchronize()
        names = ("qdot_flat", "lambda", "link_velocity_pseudo", "qdot_pseudo", "env_status", "vbd_velocity_sweep_count", "solver_residual")
        after[sick] = {name: world.download(name).reshape(count, -1) for name in names}
        if sick:
            live = (flags & 0b1001 == 1).sum(1)
            status = after[sick]["env_status"][:, 0]
            flagged = status & (1 << 13) != 0
            touching = after[False]["lambda"].any(1)
            assert flagged[chosen[kind == 0]].all() and flagged[chosen[kind == 1]].all()
            most = world.info.contact_slots_per_env * (4 if case == "box" else 2)
            assert np.array_equal(flagged[crowd], live[crowd] > most) and flagged[crowd].any() and touching.mean() > 0.3
            assert np.array_equal(np.flatnonzero(flagged), np.sort(chosen[flagged[chosen]]))
        world.close()
    others = np.setdiff1d(np.arange(count), np.arange(0, count, 5))
    assert not after[False]["env_status"].any()
    for name, value in after[False].items():
        assert np.array_equal(value[others], after[True][name][others]), name
