"""Worlds under the pyramidal cone of the compliant contact law, where a contact point is four heads of the solve."""
import copy

import numpy as np
import pytest

from test_gpu_properties import abi, nk, per_env_error

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows,cols,bounds", [(7, 6, (14, 28, 42)), (3, 5, (14, 15, 15)), (2, 2, (4, 4, 4))])
def test_environments_on_either_side_of_the_edge_capacities_match_the_oracle(oracle_py, device, rows, cols, bounds):
    """A raft of spheres over the plane, tilted or level: with 42 of them (168 heads) the solve sends environments of up to
    14, of up to 28 and of more contact points to three launches of their own; with 15, whose 60 heads leave a compute unit
    seven blocks of eight, and with four all go to one.  An environment's result is the oracle's, which knows no launches."""
    E = 96
    t = abi.Template()
    t.contact_cone = abi.CONE_PYRAMIDAL
    t.add_link(abi.JOINT_FLOATING, None, mass=5.0, diag_inertia=(0.2, 0.2, 0.4))
    profile = t.add_profile(0.7)
    for entry in t.profiles:
        entry["law"] = abi.LAW_MUJOCO
    t.add_body(abi.ROLE_STATIC, kind=abi.SHAPE_PLANE, contype=2, conaffinity=1, profile=profile)
    t.add_body(abi.ROLE_LINK_BODY, link=0, contype=0, conaffinity=0)
    for i in range(rows):
        for j in range(cols):
            t.add_body(abi.ROLE_PROXY, link=0, kind=abi.SHAPE_SPHERE, params=(0.02, 0, 0, 0), contype=1, conaffinity=2, profile=profile,
                       local_pos=(0.07 * (i - (rows - 1) / 2), 0.07 * (j - (cols - 1) / 2), 0.0))
    g = np.random.default_rng(8)
    tilt = np.concatenate([np.zeros(16), np.linspace(0.0005, 0.02, 64), g.uniform(0.02, 0.12, 16)])
    height = 0.02 * np.cos(tilt) + 0.07 * (cols - 1) / 2 * np.sin(tilt) - 0.001
    base = np.stack([g.normal(0, 0.1, E), g.normal(0, 0.1, E), height, np.cos(tilt / 2), np.sin(tilt / 2), 0 * tilt, 0 * tilt], 1)
    state = dict(q=np.zeros((E, 1), np.float32), qdot=np.zeros((E, 1), np.float32), tau=np.zeros((E, 1), np.float32),
                 base_pose=base.astype(np.float32), root_twist=(g.normal(0, 0.2, (E, 6)) * [1, 1, 1, 1, 1, 0.2]).astype(np.float32))
    desc = abi.world_desc(E, 1.0 / 200.0, vel_iters=8)
    world, oracle = nk.World(device, t, desc), oracle_py.OracleWorld(t, desc, threads=8)
    for w in (world, oracle):
        w.set_state(state)
        w.step()
    world.synchronize()
    counts = oracle.download("contact_count")
    small, middle, full = bounds
    assert counts.max() == full and (counts <= small).any() and (middle in (small, full) or ((counts > small) & (counts <= middle)).any()), np.sort(counts)
    for name in ("contact_count", "row_count", "env_status"):
        assert np.array_equal(world.download(name), oracle.download(name)), name
    assert not world.download("env_status").any()
    # single precision with up to 168 heads an environment; the bar of the native-law raft, a step instead of two
    for name in ("qdot", "link_velocity", "base_pose"):
        error = per_env_error(world.download(name), oracle.download(name), E)
        assert error.max() <= 2e-4, (name, float(error.max()), int(counts[error.argmax()]))


@pytest.mark.parametrize("E", [6144, 11519, 11520])
def test_as_many_launches_as_the_environments_pay_for_give_the_same_bits(device, E):
    """Humanoids go to one launch of five blocks a compute unit below nine rounds of 1280, and from there on to one of twelve for
    those of few contact points ahead of it: copies of 48 environments have the bits that the 48 have alone."""
    cfg = nk.synthetic.config(3, 48)
    template, state = copy.deepcopy(cfg.template), cfg.state()
    template.contact_cone = abi.CONE_PYRAMIDAL
    for profile in template.profiles:
        profile["law"] = abi.LAW_MUJOCO
    out = []
    for rows in (np.arange(48), np.arange(E) % 48):
        world = nk.World(device, template, abi.world_desc(len(rows), cfg.dt, vel_iters=cfg.vel_iters))
        world.set_state({name: values[rows] for name, values in state.items()})
        world.step()
        world.synchronize()
        assert not world.download("env_status").any()
        out.append({name: world.download(name).reshape(len(rows), -1) for name in ("contact_count", "qdot", "link_velocity", "lambda")})
        world.close()
    assert np.unique(out[0]["contact_count"]).size > 4
    for name, alone in out[0].items():
        assert np.array_equal(alone[np.arange(E) % 48], out[1][name]), name
