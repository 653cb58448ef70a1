"""Serial chains of up to eight links without rows, a lane an environment from a batch on: a step against the general kernels' ops
and, with them, against the double-precision oracle.  The one-lane walk's results are its own in their last places; below its batch a
step is the ops', bit for bit."""
import numpy as np
import pytest

from conftest import nk, relative_error

abi = nk.abi
pytestmark = pytest.mark.gpu
FIELDS = ("m", "m_factor", "articulation_bias", "articulation_qdd", "qdot", "qddot", "q", "link_velocity", "link_acceleration", "link_pose", "body_pose")
OPS = ("FkWorldPoses", "ApplyDrives", "ArticulationDynamics", "IntegrateVelocity", "IntegratePosition", "FkWorldPoses", "FkLinkVelocities", "SyncLinkBodyPose")


def chain(links, kinds, g, flat=None):
    """`links` links one on the other, the joints' types in turn `kinds`; frames, axes, inertias and the joints' own terms in general
    position.  Link `flat` has an axis of zeros."""
    t = abi.Template()
    for k in range(links):
        rotation = g.normal(size=4)
        kind = kinds[k % len(kinds)]
        t.add_link(kind, k - 1 if k else None, axis=(0, 0, 0) if k == flat else tuple(g.normal(size=3)), local_pos=tuple(g.normal(0.0, 0.15, 3)), local_rot=tuple(rotation / np.linalg.norm(rotation)),
                   mass=g.uniform(0.2, 2.0), diag_inertia=tuple(g.uniform(2e-3, 2e-2, 3)), com=tuple(g.normal(0.0, 0.05, 3)), damping=g.uniform(0.05, 0.3),
                   armature=g.uniform(0.01, 0.05), stiffness=g.uniform(0.2, 1.0), spring_ref=g.normal(0.0, 0.5))
    for link in range(links):
        t.add_body(abi.ROLE_LINK_BODY, link=link, kind=abi.SHAPE_NONE, contype=0, conaffinity=0)
    return t


R, P, F = abi.JOINT_REVOLUTE, abi.JOINT_PRISMATIC, abi.JOINT_FIXED


def fewest(links):
    """The batch from which a chain of so many links is a lane an environment."""
    return 64 if links <= 6 else 256 * (links - 6) + 1


@pytest.mark.parametrize("links,kinds", [(1, (R,)), (1, (P,)), (2, (F, R)), (5, (P, R)), (7, (R, P, F)), (8, (F, R, R, R, R, R, R, R)), (8, (R,)), (8, (R, F, P))])
@pytest.mark.parametrize("E,wrench", [(64, True), (65, False), (333, True)])
def test_a_chain_steps_like_the_ops_and_as_near_the_double_step(oracle_py, device, links, kinds, E, wrench):
    """Two steps, from the fewest environments on.  A field of the one-lane walk is within single precision's rounding over eight links of
    the general kernels' (they differ in fused products and the order of sums: 1e-5 of the field's norm, ten times what is seen; what
    follows from the accelerations within what two factorings of n coordinates may differ by, 2 n cond(M) 2^-24, where that is more), and
    no further than 1.5 times as far from the double-precision step, or under 5e-7 of the norm, where single values' last places decide."""
    E = E - 64 + fewest(links)
    g = np.random.default_rng(10 * links + len(kinds))
    t = chain(links, kinds, g, flat=3 if links == 5 else None)
    jointed = np.array([link["joint_type"] != F for link in t.links])
    state = {name: (g.normal(0.0, sigma, (E, links)) * jointed).astype(np.float32) for name, sigma in (("q", 1.0), ("qdot", 1.0), ("tau", 2.0))}
    base = g.normal(size=(E, 7)).astype(np.float32)   # (of no concern to a root that stands still)
    base[:, 3:] /= np.linalg.norm(base[:, 3:], axis=1, keepdims=True)
    state.update(base_pose=base, root_twist=np.zeros((E, 6), np.float32))
    gravity_force = g.normal(0.0, 1.0, (E, links)).astype(np.float32)
    pushes = g.normal(0.0, 1.0, (E, links, 6)).astype(np.float32) * (g.random((E, links, 1)) < 0.2)
    desc = abi.world_desc(E, 1.0 / 240.0)
    worlds = [nk.World(device, t, desc), nk.World(device, t, desc), oracle_py.OracleWorld(t, desc, threads=4, double=True)]
    out = []
    for kind, w in zip(("ops", "step", "double"), worlds):
        w.set_state(state)
        w.upload("joint_gravity_force", gravity_force)
        for _ in range(2):
            if wrench:
                w.upload("link_wrench", pushes)
            if kind == "ops":
                for op in OPS:
                    w.op(op)
            else:
                w.step()
        if kind != "double":
            w.synchronize()
        if kind == "step":
            assert not np.any(w.download("link_wrench"))
        out.append({name: w.download(name).astype(np.float64).reshape(E, -1) for name in FIELDS if kind != "double" or name not in ("m_factor", "body_pose")})
        w.close()
    ops, step, double = out
    assert links < 5 or any(not np.array_equal(step[name], ops[name]) for name in FIELDS)   # the one-lane walk's
    assert np.abs(ops["articulation_qdd"]).max() > 0.1 and np.isfinite(step["link_pose"]).all()
    n = int(jointed.sum())
    solved = 2 * n * np.linalg.cond(double["m"].reshape(E, n, n)).max() * 2.0 ** -24
    for name in FIELDS:
        bound = 1e-5 if name in ("m", "m_factor", "articulation_bias") else max(1e-5, solved)
        assert relative_error(step[name], ops[name]) <= bound, (name, relative_error(step[name], ops[name]), bound)
        if name in double:
            scale = np.linalg.norm(double[name]) + 1e-30
            mine, general = np.linalg.norm(step[name] - double[name]) / scale, np.linalg.norm(ops[name] - double[name]) / scale
            assert mine <= max(1.5 * general, 5e-7), (name, mine, general)


@pytest.mark.parametrize("links,E", [(1, 63), (6, 63), (7, 64), (7, 256), (8, 512)])
def test_below_its_batch_a_step_is_the_ops(device, links, E):
    """The general kernels in one launch and one by one, and the environments of a smaller batch among a larger's."""
    t = chain(links, (R, P, R), np.random.default_rng(links))
    g = np.random.default_rng(E)
    state = {name: g.normal(0.0, 1.0, (E, links)).astype(np.float32) for name in ("q", "qdot", "tau")}
    base = np.zeros((E, 7), np.float32)
    base[:, 3] = 1.0
    state.update(base_pose=base, root_twist=np.zeros((E, 6), np.float32))
    out = []
    for kind, envs in (("ops", E), ("step", E), ("step", 17)):
        w = nk.World(device, t, abi.world_desc(envs, 1.0 / 240.0))
        w.set_state({name: v[:envs] for name, v in state.items()})
        for _ in range(2):
            if kind == "ops":
                for op in OPS:
                    w.op(op)
            else:
                w.step()
        w.synchronize()
        out.append({name: w.download(name).reshape(envs, -1) for name in FIELDS})
        w.close()
    for name in FIELDS:
        assert np.array_equal(out[0][name].view(np.uint8), out[1][name].view(np.uint8)), name
        assert np.array_equal(out[2][name].view(np.uint8), out[1][name][:17].view(np.uint8)), name


@pytest.mark.parametrize("kinds", [(R, F, P, R, F), (F, P, R, F, R, R, P, F)])
def test_a_coordinate_counts_where_its_joint_has_a_use_for_it(device, kinds):
    """A fixed link's coordinate that is not finite reaches its own word and nothing else; a joint's reaches what it reaches in the
    general kernels' ops."""
    links = len(kinds)
    E = fewest(links) + 6
    g = np.random.default_rng(links)
    t = chain(links, kinds, g)
    jointed = np.array([kind != F for kind in kinds])
    state = {name: (g.normal(0.0, sigma, (E, links)) * jointed).astype(np.float32) for name, sigma in (("q", 1.0), ("qdot", 1.0), ("tau", 2.0))}
    base = np.zeros((E, 7), np.float32)
    base[:, 3] = 1.0
    state.update(base_pose=base, root_twist=np.zeros((E, 6), np.float32))
    fixed, moving = np.flatnonzero(~jointed), np.flatnonzero(jointed)
    for env, value in ((3, np.nan), (5, np.inf), (9, -np.inf), (69, np.nan)):
        state["q"][env, fixed] = value
    for k, link in enumerate(moving):
        state["q"][20 + 2 * k, link], state["q"][21 + 2 * k, link] = np.inf, np.nan
    out = []
    for kind in ("ops", "step"):
        w = nk.World(device, t, abi.world_desc(E, 1.0 / 240.0))
        w.set_state(state)
        if kind == "ops":
            for op in OPS:
                w.op(op)
        else:
            w.step()
        w.synchronize()
        out.append({name: w.download(name).astype(np.float64).reshape(E, -1) for name in FIELDS})
        w.close()
    ops, step = out
    for name in FIELDS:
        assert np.array_equal(np.isfinite(step[name]), np.isfinite(ops[name])), name
        unused = np.zeros(links, bool) if name != "q" else ~jointed
        assert np.isfinite(step[name][[3, 5, 9, 69]][:, ~np.resize(unused, step[name].shape[1])]).all(), name
        whole = np.isfinite(ops[name])
        assert relative_error(step[name][whole], ops[name][whole]) <= 1e-5, name


@pytest.mark.parametrize("bodies", [3, 70, 300])
def test_a_chains_bodies_follow_their_links(device, bodies):
    """Rows that follow a link as they are, from a place of their own on it, and rows that stand still, more of them than lanes and than
    a workgroup has: the ops' poses, and the cooked ones where nothing moves."""
    E, links = 70, 5
    g = np.random.default_rng(bodies)
    t = chain(links, (R, P, F, R), g)
    roles = g.integers(0, 3, bodies)
    for role in roles:
        place = dict(kind=abi.SHAPE_SPHERE, params=(0.1, 0, 0, 0), local_pos=tuple(g.normal(size=3)), contype=0, conaffinity=0)
        if role == 0:
            t.add_body(abi.ROLE_STATIC, **place)
        else:
            t.add_body(abi.ROLE_PROXY, link=int(g.integers(links)), **place)
    jointed = np.array([link["joint_type"] != F for link in t.links])
    state = {name: (g.normal(0.0, 1.0, (E, links)) * jointed).astype(np.float32) for name in ("q", "qdot", "tau")}
    base = np.zeros((E, 7), np.float32)
    base[:, 3] = 1.0
    state.update(base_pose=base, root_twist=np.zeros((E, 6), np.float32))
    out = []
    for kind in ("ops", "step"):
        w = nk.World(device, t, abi.world_desc(E, 1.0 / 240.0))
        w.set_state(state)
        before = w.download("body_pose").reshape(E, -1, 7)
        if kind == "ops":
            for op in OPS:
                w.op(op)
        else:
            w.step()
        w.synchronize()
        out.append(w.download("body_pose").reshape(E, -1, 7).astype(np.float64))
        w.close()
    ops, step = out
    still = np.concatenate([np.zeros(links, bool), roles == 0])
    assert np.array_equal(step[:, still], before[:, still]) and not np.array_equal(step[:, ~still], before[:, ~still])
    assert relative_error(step, ops) <= 1e-5
