"""The solve's launch order: every environment once, and in a state its history says nothing of, those whose free velocity
drives into more contact points first."""
import numpy as np
import pytest

from conftest import nk

pytestmark = pytest.mark.gpu
abi = nk.abi


@pytest.mark.parametrize("index,E", [(2, 1), (2, 1023), (2, 1025), (3, 257), (6, 4097), (6, 8195)])
def test_environments_that_land_come_ahead_of_those_in_the_air(device, index, E):
    cfg = nk.synthetic.config(index, E)
    world = nk.World(device, cfg.template, abi.world_desc(E, cfg.dt, vel_iters=cfg.vel_iters))
    state = cfg.state()
    standing = np.arange(E) % 3 == 1
    aloft = {name: values.copy() for name, values in state.items()}
    aloft["base_pose"][:, 2] += 5.0
    world.set_state(aloft)
    world.step()
    world.synchronize()
    assert not world.download("contact_count").any()
    assert np.array_equal(np.sort(world.download("tile_order")), np.arange(E))
    mixed = {name: values.copy() for name, values in state.items()}
    mixed["base_pose"][~standing, 2] += 5.0
    world.set_state(mixed)
    world.step()
    world.synchronize()
    order, points = world.download("tile_order"), world.download("solver_points") >> 16
    assert np.array_equal(np.sort(order), np.arange(E))
    assert not points[~standing].any() and (points[standing] <= world.download("contact_count")[standing]).all()
    if standing.any():
        assert (points[standing] > 0).mean() > 0.5
    blocks = (E + 1023) // 1024   # each sorts every blocks-th environment
    for first in range(blocks):
        landing = points[order[first::blocks]] > 0 if blocks > 1 else points[order] > 0
        assert not (landing[1:] & ~landing[:-1]).any()
    world.close()


@pytest.mark.parametrize("index,E", [(2, 300), (3, 300), (6, 8200)])
def test_the_work_field_holds_the_decaying_maximum_of_the_solves(device, index, E):
    """solver_cost is the work of the last solve or three quarters of what stood there, whichever is more, over the whole range of
    the word; the order goes by it in a state that was solved before."""
    cfg = nk.synthetic.config(index, E)
    world = nk.World(device, cfg.template, abi.world_desc(E, cfg.dt, vel_iters=cfg.vel_iters))
    world.set_state(cfg.state())
    start = world.checkpoint()
    world.restore(start)
    world.step()
    world.synchronize()
    work = world.download("solver_cost").astype(np.int64)
    assert work.any() and work.max() < 1 << 16
    earlier = np.random.default_rng(E).integers(0, 1 << 32, E, dtype=np.int64) >> np.arange(E) % 24 | 1
    world.upload("solver_cost", earlier.astype(np.uint32))
    world.restore(start)
    world.step()
    world.synchronize()
    assert np.array_equal(world.download("solver_cost"), np.maximum(work, earlier - earlier // 4))
    order, points = world.download("tile_order"), world.download("solver_points")
    assert np.array_equal(points & 0xFFFF, points >> 16)
    blocks = (E + 1023) // 1024
    for first in range(blocks):
        mine = order[first::blocks]
        level = earlier[mine] // (earlier[mine].max() // 256 + 1)
        assert (mine % blocks == first).all() and (np.diff(level) <= 0).all()
    world.close()


@pytest.mark.parametrize("index,law", [(2, "native"), (3, "native"), (2, "elliptic"), (3, "elliptic"), (2, "pyramidal"), (3, "pyramidal")])
def test_the_counted_points_are_those_whose_first_row_the_free_velocity_drives_into(device, index, law):
    """By the rows as the solve meets them: a compliant row's right-hand side includes the damping of the start velocity."""
    E = 200
    cfg = nk.synthetic.config(index, E)
    if law != "native":
        for profile in cfg.template.profiles:
            profile["law"] = abi.LAW_MUJOCO
        cfg.template.contact_cone = abi.CONE_ELLIPTIC if law == "elliptic" else abi.CONE_PYRAMIDAL
    world = nk.World(device, cfg.template, abi.world_desc(E, cfg.dt, vel_iters=cfg.vel_iters))
    world.set_state(cfg.state())
    world.step()
    world.synchronize()
    R, S, md = world.rows_per_env, world.info.contact_slots_per_env, world.download("solver_free").size // E
    words = world.download("urows").reshape(E, R, -1)
    ranges = world.download("ucontact_row_range").reshape(E, S, 2).astype(np.int64)
    jacobian = (world.download("chain_jacobian").reshape(E, R, md) + world.download("chain_jacobian_b").reshape(E, R, md)).astype(np.float64)
    free = world.download("solver_free").reshape(E, md).astype(np.float64)
    expect, clear = np.zeros(E, np.int64), np.ones(E, bool)
    for env in range(E):
        for first, count in ranges[env] - np.array([env * R, 0]):
            for row in range(first, first + count):
                if not words[env, row, 0].view(np.uint32) & 1:
                    continue
                terms = jacobian[env, row] * free[env]
                gap = float(words[env, row, 4]) * cfg.dt - terms.sum()
                expect[env] += gap > 0.0
                clear[env] &= abs(gap) > 1e-5 * (1.0 + np.abs(terms).sum())   # (64 terms in single precision: below 64 / 2^24 of their size)
    assert clear.mean() > 0.9 and expect.any()
    assert np.array_equal((world.download("solver_points") >> 16)[clear], expect[clear])
    world.close()


@pytest.mark.parametrize("law", ["native", "pyramidal"])
def test_a_new_state_is_ordered_by_its_points_but_under_the_pyramidal_cone(device, law):
    """There the points say little of a solve's length: the order stays that of the work."""
    E = 300
    cfg = nk.synthetic.config(2, E)
    if law == "pyramidal":
        for profile in cfg.template.profiles:
            profile["law"] = abi.LAW_MUJOCO
        cfg.template.contact_cone = abi.CONE_PYRAMIDAL
    world = nk.World(device, cfg.template, abi.world_desc(E, cfg.dt, vel_iters=cfg.vel_iters))
    world.set_state(cfg.state())
    work = (np.random.default_rng(7).permutation(E) + 1) * 16
    world.upload("solver_cost", work.astype(np.uint32))
    world.upload("solver_points", np.full(E, 0xFFFF, np.uint32))   # no state has so many
    world.step()
    world.synchronize()
    order, points = world.download("tile_order"), world.download("solver_points") >> 16
    assert np.array_equal(np.sort(order), np.arange(E)) and len(np.unique(points)) > 2
    by = work if law == "pyramidal" else points
    level = by[order].astype(np.int64) // (work.max() // 256 + 1 if law == "pyramidal" else 1)
    assert (np.diff(level) <= 0).all()
    world.close()
