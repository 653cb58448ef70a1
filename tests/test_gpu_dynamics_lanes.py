"""The forward dynamics at its lane counts: 64 lanes an environment for small batches and large robots, 16 or 8 for large
batches of small ones; and the launches that take the poses and the step's tail with it."""
import numpy as np
import pytest

from conftest import nk, relative_error
from trees import tree_case

abi = nk.abi
pytestmark = pytest.mark.gpu
FIELDS = ("m", "m_factor", "articulation_bias", "articulation_qdd", "qdot", "qddot", "link_velocity", "link_acceleration", "link_wrench")


def dynamics(device, tree, state, rows):
    E = len(rows)
    world = nk.World(device, tree.template, abi.world_desc(E, 1.0 / 240.0, vel_iters=8, contact_margin=0.1))
    world.set_state({k: v[rows] for k, v in state.items()})
    world.op("FkWorldPoses")
    world.op("ArticulationDynamics")
    world.synchronize()
    out = {name: world.download(name).reshape(E, -1) for name in FIELDS}
    world.close()
    return out


@pytest.mark.parametrize("dof,floating,branched,limb_joints,links", [
    (1, False, False, 7, 2),     # eight lanes: one joint,
    (7, False, False, 7, 8),     # a chain, a link a step,
    (7, False, True, 1, 8),      # seven links of one depth, a step each,
    (13, True, False, 7, 8),     # more coordinates than links
    (8, False, False, 7, 9),     # sixteen lanes: the fewest links,
    (15, False, True, 1, 16),    # fifteen links of one depth, in passes of ten and steps of two,
    (21, True, True, 4, 16),     # the most links and coordinates of a floating robot
    (16, False, True, 3, 17),    # sixty-four lanes whatever the batch
])
@pytest.mark.parametrize("E", [1152, 2560, 3077])
def test_packed_environments_have_the_bits_they_have_alone(oracle_py, device, dof, floating, branched, limb_joints, links, E):
    """From 1152 environments of up to eight links on, and 2560 of up to sixteen, a workgroup takes eight or four of them; the
    arithmetic is the same, so copies of 48 seeded environments give in every place, also in a last workgroup that is not full,
    the bits that the 48 give alone."""
    tree, _, state = tree_case(oracle_py, dof, floating, branched, seed=3 * dof + 1, E=48, limb_joints=limb_joints)
    assert tree.link_count == links
    rows = np.arange(E) % 48
    alone, packed = dynamics(device, tree, state, np.arange(48)), dynamics(device, tree, state, rows)
    assert np.abs(alone["articulation_qdd"]).max() > 0.1
    for name in FIELDS:
        assert np.array_equal(alone[name][rows], packed[name]), name


@pytest.mark.parametrize("links", [64, 65, 128, 129, 150])
def test_many_links_match_the_oracle(oracle_py, device, links):
    """A lane takes two links of the mass matrix up to 128 of them, whose matrix then stands where their inertias did; past
    that the two stand apart.  Twelve joints among links fixed to one another, in limbs of equal length."""
    E, g = 32, np.random.default_rng(links)
    t = abi.Template()
    t.add_link(abi.JOINT_FLOATING, None, mass=4.0, diag_inertia=(0.05, 0.06, 0.07))
    limb, parents = (links - 1 + 2) // 3, [0, 0, 0]
    for k in range(links - 1):
        side, hinge = k // limb, k % limb in (0, 2, limb // 2, limb - 2)
        parents[side] = t.add_link(abi.JOINT_REVOLUTE if hinge else abi.JOINT_FIXED, parents[side], axis=((1, 0, 0), (0, 1, 0), (0, 0, 1))[k % 3],
                                   local_pos=(0.02 * (side - 1), 0.01, -0.03), mass=g.uniform(0.02, 0.2),
                                   diag_inertia=tuple(g.uniform(1e-4, 5e-4, 3)), com=(0.0, 0.0, -0.01), armature=0.02)
    for link in range(t.link_count):
        t.add_body(abi.ROLE_LINK_BODY, link=link, kind=abi.SHAPE_NONE, contype=0, conaffinity=0)
    base = np.zeros((E, 7), np.float32)
    base[:, 3] = 1.0
    base[:, 4:] = 0.5 * g.normal(0.0, 0.2, (E, 3))
    base[:, 3:] /= np.linalg.norm(base[:, 3:], axis=1, keepdims=True)
    hinges = np.array([link["joint_type"] == abi.JOINT_REVOLUTE for link in t.links])
    state = {name: (g.normal(0.0, sigma, (E, links)) * hinges).astype(np.float32) for name, sigma in (("q", 0.3), ("qdot", 0.5), ("tau", 0.5))}
    state.update(base_pose=base, root_twist=g.normal(0.0, 0.3, (E, 6)).astype(np.float32))
    desc = abi.world_desc(E, 1.0 / 240.0)
    world, oracle = nk.World(device, t, desc), oracle_py.OracleWorld(t, desc, threads=4)
    assert world.link_count == links
    for w in (world, oracle):
        w.set_state(state)
        w.step()
    world.synchronize()
    # a chain of some fifty links sums in another order than the oracle's nowhere; single precision over its depth
    for name, bar in (("m", 2e-6), ("articulation_bias", 5e-6), ("articulation_qdd", 5e-5), ("qdot", 5e-5), ("link_acceleration", 5e-5)):
        error = relative_error(world.download(name), oracle.download(name))
        assert error <= bar, (name, error)
    world.close()
    oracle.close()


@pytest.mark.parametrize("dof,floating,branched,limb_joints,E", [
    (16, False, True, 3, 1), (16, False, True, 3, 1536), (16, False, True, 3, 1537),   # a wavefront each: one, the most, one more
    (7, False, False, 7, 48), (7, False, False, 7, 3077),                              # a chain alone, and eight a workgroup
    (21, True, True, 4, 1000), (21, True, True, 4, 3077),                              # a floating robot alone, and four a workgroup
])
def test_poses_beside_the_dynamics_are_those_ahead_of_it(oracle_py, device, dof, floating, branched, limb_joints, E):
    """A step places the links in the dynamics' launch, where a link with a wrench on it turns that by its own new pose: the
    state after the step has the bits the ops leave one by one, from poses and wrenches that were uploaded."""
    tree, _, state = tree_case(oracle_py, dof, floating, branched, seed=dof, E=48, limb_joints=limb_joints)
    rows, g = np.arange(E) % 48, np.random.default_rng(dof)
    nl = tree.link_count
    wrench = g.normal(0.0, 2.0, (E, nl, 6)).astype(np.float32) * (g.random((E, nl, 1)) < 0.3)
    out = []
    for single in (True, False):
        world = nk.World(device, tree.template, abi.world_desc(E, 1.0 / 240.0, vel_iters=8, contact_margin=0.1))
        world.set_state({k: v[rows] for k, v in state.items()})
        world.upload("link_pose", np.full((E, nl, 7), np.nan, np.float32))
        world.upload("link_wrench", wrench)
        if single:
            for op in ("FkWorldPoses", "ApplyDrives", "ArticulationDynamics", "SyncLinkBodyPose", "BuildAabbs", "LbvhBuild", "LbvhQueryPairs",
                       "NarrowphasePrimitives", "AssembleRows", ("ContactWarmStart", 0), "BlockDescentSolve", ("ContactWarmStart", 1),
                       "IntegratePosition", "FkWorldPoses", "FkLinkVelocities", "SyncLinkBodyPose"):
                world.op(*(op if isinstance(op, tuple) else (op,)))
        else:
            world.step()
        world.synchronize()
        out.append({name: world.download(name).reshape(E, -1) for name in FIELDS + ("q", "link_pose")})
        world.close()
    assert np.abs(out[0]["articulation_qdd"]).max() > 0.1 and np.isfinite(out[0]["qddot"]).all()
    for name in out[0]:
        assert np.array_equal(out[0][name], out[1][name]), name


@pytest.mark.parametrize("links,E", [(2, 1), (8, 48), (8, 3077), (8, 10240), (8, 10241), (17, 1280), (17, 1281)])
def test_a_step_without_rows_is_one_launch_with_the_bits_of_its_ops(device, links, E):
    """A world without rows goes on from the dynamics to the step's tail in the same workgroup, up to 1280 of them: the state after
    two steps, the second from poses and twists the first left, has the bits the ops leave one by one."""
    g = np.random.default_rng(links)
    t = abi.Template()
    t.add_link(abi.JOINT_FIXED, None, mass=2.0, diag_inertia=(0.02, 0.03, 0.02))
    for k in range(links - 1):
        t.add_link(abi.JOINT_REVOLUTE, max(0, k - k % 3 // 2), axis=((1, 0, 0), (0, 1, 0), (0, 0, 1))[k % 3], local_pos=(0.1, 0.02, -0.05),
                   mass=g.uniform(0.1, 0.5), diag_inertia=tuple(g.uniform(1e-3, 5e-3, 3)), com=(0.0, 0.01, -0.03), armature=0.02)
    for link in range(t.link_count):
        t.add_body(abi.ROLE_LINK_BODY, link=link, kind=abi.SHAPE_NONE, contype=0, conaffinity=0)
    rows = np.arange(E) % 48
    state = {name: g.normal(0.0, sigma, (48, links)).astype(np.float32)[rows] for name, sigma in (("q", 0.5), ("qdot", 1.0), ("tau", 0.5))}
    base = np.zeros((E, 7), np.float32)
    base[:, 3] = 1.0
    state.update(base_pose=base, root_twist=np.zeros((E, 6), np.float32))
    for name in ("q", "qdot", "tau"):
        state[name][:, 0] = 0.0
    wrench = g.normal(0.0, 0.5, (48, links, 6)).astype(np.float32)[rows]
    out = []
    for single in (True, False):
        world = nk.World(device, t, abi.world_desc(E, 1.0 / 240.0))
        world.set_state(state)
        for _ in range(2):
            world.upload("link_wrench", wrench)
            if single:
                for op in ("FkWorldPoses", "ApplyDrives", "ArticulationDynamics", "IntegrateVelocity", "IntegratePosition", "FkWorldPoses", "FkLinkVelocities", "SyncLinkBodyPose"):
                    world.op(op)
            else:
                world.step()
        world.synchronize()
        out.append({name: world.download(name).reshape(E, -1) for name in FIELDS + ("q", "link_pose", "body_pose")})
        world.close()
    assert np.isfinite(out[0]["link_pose"]).all() and np.abs(out[0]["qdot"]).max() > 0.1
    for name in out[0]:
        assert np.array_equal(out[0][name], out[1][name]), name
