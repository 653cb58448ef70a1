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
