"""Candidate pairs: the walk over pairs of rows at the edges of its passes of 64, with exclusions in LDS and in memory."""
import numpy as np
import pytest

from conftest import nk

abi = nk.abi
pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows,excluded", [(1, 0.0), (2, 0.0), (2, 1.0), (11, 0.3), (12, 0.0), (12, 0.3), (17, 0.5), (34, 0.85), (34, 0.97)])
def test_pairs_are_the_overlapping_ones_in_ascending_order(device, rows, excluded):
    """Spheres on sliders of their own: 1 and 2 rows, 55 and 66 pairs (a pass is 64), 561 with fewer and with more exclusions than
    LDS holds (512).  The one launch ahead of the row assembly and the ops one by one give the pairs of the boxes, exactly."""
    g, E = np.random.default_rng(rows), 96
    t = abi.Template()
    t.add_link(abi.JOINT_FIXED, None, mass=1.0)
    profile = t.add_profile(0.5)
    for k in range(rows):
        link = t.add_link(abi.JOINT_PRISMATIC, 0, axis=((1, 0, 0), (0, 1, 0), (0, 0, 1))[k % 3], mass=0.3, diag_inertia=(0.002, 0.003, 0.0025))
        t.add_body(abi.ROLE_LINK_BODY, link=link, kind=abi.SHAPE_SPHERE, params=(0.05, 0, 0, 0), contype=1, conaffinity=1, profile=profile)
    pairs = [(i, j) for i in range(rows) for j in range(i + 1, rows)]
    out = [pair for pair in pairs if g.random() < excluded]
    if rows == 34:
        assert (len(out) > 512) == (excluded > 0.95)
    for pair in out:
        t.exclude(*pair)
    t.max_contacts_per_env = 24
    q = g.normal(0.0, 0.1, (E, rows + 1)).astype(np.float32)
    q[:, 0] = 0.0
    zeros, base = np.zeros((E, rows + 1), np.float32), np.tile([0, 0, 0, 1, 0, 0, 0], (E, 1)).astype(np.float32)
    results = []
    for single in (True, False):
        world = nk.World(device, t, abi.world_desc(E, 1.0 / 240.0, contact_margin=0.01))
        world.set_state(dict(q=q, qdot=zeros, tau=zeros, base_pose=base, root_twist=np.zeros((E, 6), np.float32)))
        if single:
            for op in ("FkWorldPoses", "SyncLinkBodyPose", "BuildAabbs", "LbvhBuild", "LbvhQueryPairs"):
                world.op(op)
        else:
            world.step()
        world.synchronize()
        results.append({name: world.download(name) for name in ("body_aabb_lo", "body_aabb_hi", "candidate_pairs", "pair_count")})
        results[-1]["overflow"] = world.download("env_status") if single else None
        world.close()
    lo, hi = (results[0][name].reshape(E, -1, 3) for name in ("body_aabb_lo", "body_aabb_hi"))
    assert lo.shape[1] == rows
    gone, seen = set(out), 0
    for e in range(E):
        expect = [(i, j) for i, j in pairs if (i, j) not in gone and not ((hi[e, i] < lo[e, j]) | (lo[e, i] > hi[e, j])).any()]
        seen += len(expect)
        for r in results:
            count = int(r["pair_count"][e])
            assert count == min(len(expect), 24)
            assert [tuple(p) for p in r["candidate_pairs"].reshape(E, -1, 2)[e, :count]] == expect[:24]
        assert (results[0]["overflow"][e] != 0) == (len(expect) > 24)
    assert seen > 0 or len(out) == len(pairs)
    for name in ("body_aabb_lo", "body_aabb_hi"):
        assert np.array_equal(results[0][name].view(np.uint32), results[1][name].view(np.uint32))
