"""Contact rows after a restore, and the readout over them: the row assembly clears what the world's own steps left in
memory, whatever extent a checkpoint brings back, and the readout takes the rows of the last step, 64 at a time."""
import os

import numpy as np
import pytest

from conftest import ROOT, nk

abi = nk.abi
pytestmark = pytest.mark.gpu
WALKER = os.path.join(ROOT, "tests", "data", "capsule_walker.xml")
ROWS = ("row_count", "contact_count", "contact_row_extent", "row_cj_link", "row_cj_link_b", "row_penetration", "lambda", "link_contact_wrench",
        "q", "qdot", "env_status")


def made(device, robot, envs):
    """(world, time step, state on the ground, state out of its reach)"""
    if robot == "walker":
        scene = nk.Scene(WALKER)
        dt = scene.info.timestep
        world = nk.World(device, scene, abi.world_desc(envs, dt, vel_iters=8))
        rest = np.zeros((envs, scene.link_count), np.float32)
        low = dict(q=rest, qdot=rest, tau=rest, base_pose=np.tile(np.array([0, 0, 0.54, 1, 0, 0, 0], np.float32), (envs, 1)),
                   root_twist=np.zeros((envs, 6), np.float32))
    else:
        cfg = nk.synthetic.config({"quadruped": 2, "rope": 5}[robot], envs)
        dt = cfg.dt
        world = nk.World(device, cfg.template, abi.world_desc(envs, dt, vel_iters=cfg.vel_iters))
        low = cfg.state()
    if robot == "rope":                                  # its root is fixed: bent upwards it leaves the plane
        high = dict(low, q=low["q"].copy())
        high["q"][:, 1] -= 1.2
    else:
        high = dict(low, base_pose=low["base_pose"].copy())
        high["base_pose"][:, 2] += 3.0
    return world, dt, low, high


def rows_of(world):
    world.synchronize()
    out = {name: world.download(name) for name in ROWS}
    out["flags"] = world.download("urows").view(np.uint32).reshape(-1, 26)[:, 0]
    return out


@pytest.mark.parametrize("graph", [False, True])
@pytest.mark.parametrize("robot,envs", [("quadruped", 65), ("rope", 33), ("walker", 65)])
def test_a_restore_leaves_no_row_of_the_steps_before_it(device, robot, envs, graph):
    world, _, low, high = made(device, robot, envs)
    fresh = made(device, robot, envs)[0]
    for w in (world, fresh):
        w.set_execution_mode(graph)
        w.download("link_contact_wrench")                # the readout joins the steps
    world.set_state(high)
    aloft = world.checkpoint()
    world.set_state(low)
    world.step(2)
    grounded = rows_of(world)
    active = (grounded["flags"].reshape(envs, -1) & 1).sum(1)
    world.restore(aloft)
    world.reset_envs([1, envs - 1, 1])                   # and environments that a reset gave no extent at all
    world.restore(aloft)
    world.step()
    fresh.set_state(high)
    fresh.step()
    after, expect = rows_of(world), rows_of(fresh)
    left = (expect["flags"].reshape(envs, -1) & 1).sum(1)
    # (some quadrupeds of the seeded batch start above the plane)
    assert (left < active).mean() > 0.75, "the restored state must hold fewer rows than the steps left"
    for name, value in expect.items():
        assert np.array_equal(after[name], value), name
    nk.lib().nuka_checkpoint_destroy(aloft)
    world.close(); fresh.close()


@pytest.mark.parametrize("robot,envs", [("quadruped", 33), ("rope", 17), ("walker", 33)])
def test_link_wrenches_are_the_sums_of_the_rows(device, robot, envs):
    """12, 192 and 304 rows an environment: less than one, three and more than four turns of 64."""
    world, dt, low, _ = made(device, robot, envs)
    world.download("link_contact_wrench")
    world.set_state(low)
    world.step(2)
    world.synchronize()
    R, nl = world.rows_per_env, world.download("q").size // envs
    rows = world.download("urows").reshape(envs, R, 26)
    active = (rows.view(np.uint32)[:, :, 0] & 1) != 0
    impulse = world.download("lambda").reshape(envs, R).astype(np.float64)
    origin = world.download("link_pose").reshape(envs * nl, 7)[:, :3].astype(np.float64)
    wrench, size = np.zeros((envs * nl, 6)), np.zeros(envs * nl)
    for side, (words, links, points) in enumerate(((slice(12, 15), "row_cj_link", "row_cj_point"), (slice(20, 23), "row_cj_link_b", "row_cj_point_b"))):
        link = world.download(links).reshape(envs, R)
        point = world.download(points).reshape(envs, R, 3).astype(np.float64)
        for e, r in zip(*np.nonzero(active & (link != abi.INVALID))):
            force = rows[e, r, words].astype(np.float64) * impulse[e, r]
            arm = point[e, r] - origin[link[e, r]]
            wrench[link[e, r]] += np.r_[force, np.cross(arm, force)]
            size[link[e, r]] += np.abs(force).max() * (1.0 + np.abs(arm).max() + np.abs(point[e, r]).max())
    got = world.download("link_contact_wrench").reshape(envs * nl, 6).astype(np.float64)
    assert active.any(1).mean() > 0.75 and np.abs(wrench).max() > 0.0
    # a row's terms round a handful of times each, and as many sums as the link has rows follow: some tens of half an ulp of their size
    assert np.all(np.abs(got - wrench / dt) <= 64 * 6e-8 / dt * size[:, None] + 1e-12)
    world.close()


@pytest.mark.parametrize("robot,envs", [("quadruped", 65), ("rope", 33), ("walker", 65)])
def test_steps_after_restores_are_those_of_a_world_never_restored(device, robot, envs):
    """From the ground to the air and back, several steps each, a plan's replays and eager steps in turn: what the rows of
    one leave behind must not reach the other."""
    world, _, low, high = made(device, robot, envs)
    world.download("link_contact_wrench")
    held, points = {}, {}
    for name, state in (("low", low), ("high", high)):
        world.set_state(state)
        held[name] = world.checkpoint()
    world.restore(held["low"])
    world.set_execution_mode(True)
    world.step(3)
    for name, state, modes in (("high", high, (False, True, True)), ("low", low, (True, False, False, True)), ("high", high, (True, False)),
                               ("low", low, (False, True))):
        world.restore(held[name])
        for graph in modes:
            world.set_execution_mode(graph)
            world.step()
        fresh = made(device, robot, envs)[0]
        fresh.download("link_contact_wrench")
        fresh.set_state(state)
        fresh.step(len(modes))
        after, expect = rows_of(world), rows_of(fresh)
        points[name] = int(expect["contact_count"].sum())
        for field, value in expect.items():
            assert np.array_equal(after[field], value), (name, modes, field)
        fresh.close()
    assert points["low"] > 2 * points["high"]
    for checkpoint in held.values():
        nk.lib().nuka_checkpoint_destroy(checkpoint)
    world.close()
