"""How far single-precision steps end from the double-precision oracle's, over enough environments that a few parts in a
hundred show."""
import copy
import os

import numpy as np
import pytest

from conftest import ROOT, nk

pytestmark = pytest.mark.gpu
abi = nk.abi
WALKER = os.path.join(ROOT, "tests", "data", "capsule_walker.xml")


class WithArrays:
    """A scene as the double-precision oracle takes a template: with the arrays behind its description."""

    def __init__(self, scene):
        self.scene, self.link_count = scene, scene.link_count

    def to_c(self):
        return self.scene.to_c()[0], self.scene.template_arrays()


def test_a_robot_files_step_is_as_near_the_double_one_as_the_oracles(oracle_py, device):
    """The walker: contact edges on one axis and joint rows beside them, an accumulation whose order shows.  The mean over
    the environments of the velocities' error is no larger than the single-precision oracle's (0.985 of it; 1.005 where the
    mass matrix was added after the sum over the heads; half a part in a hundred is what the ratio moves by between batches
    of this size)."""
    E = 32768
    scene = nk.Scene(WALKER)
    desc = abi.world_desc(E, scene.info.timestep, gravity=tuple(scene.info.gravity), vel_iters=8)
    nl, rng = scene.link_count, np.random.default_rng(11)
    q, qdot = rng.normal(0.0, 0.05, (E, nl)).astype(np.float32), rng.normal(0.0, 0.3, (E, nl)).astype(np.float32)
    q[:, 0] = qdot[:, 0] = 0.0
    base = np.zeros((E, 7), np.float32)
    base[:, 2], base[:, 3] = rng.uniform(0.53, 0.55, E), 1.0
    base[:, 4:] = rng.normal(0.0, 0.015, (E, 3))
    base[:, 3:] /= np.linalg.norm(base[:, 3:], axis=1, keepdims=True)
    state = dict(q=q, qdot=qdot, tau=np.zeros((E, nl), np.float32), base_pose=base, root_twist=rng.normal(0.0, 0.3, (E, 6)).astype(np.float32))
    authored = scene.initial_state()

    def stepped(w, on_device):
        w.set_state(state)
        if not on_device:
            for name in ("drive_stiffness", "drive_damping", "drive_force_limit", "drive_joint_force_limit"):
                w.upload(name, np.tile(authored[name], (E, 1)))
        w.upload("drive_target", np.tile(authored["q"], (E, 1)))
        w.step()
        if on_device:
            w.synchronize()
        out = w.download("link_velocity").astype(np.float64).reshape(E, -1), w.download("contact_count")
        w.close()
        return out

    got, points = stepped(nk.World(device, scene, desc), True)
    single, _ = stepped(oracle_py.OracleWorld(scene, desc, threads=8), False)
    double, expect = stepped(oracle_py.OracleWorld(WithArrays(scene), desc, threads=8, double=True), False)
    same = points == expect
    assert same.mean() > 0.99 and (points[same] > 0).mean() > 0.5
    scale = np.maximum(np.linalg.norm(double, axis=1), 1e-2)
    device_error, oracle_error = (np.linalg.norm(v - double, axis=1)[same] / scale[same] for v in (got, single))
    cap = np.quantile(oracle_error, 0.999)
    ratio = np.minimum(device_error, cap).mean() / np.minimum(oracle_error, cap).mean()
    print(f"walker: mean error {np.minimum(device_error, cap).mean():.3e}, {ratio:.4f} of the oracle's")
    assert ratio <= 1.0
    scene.close()


def elliptic(cfg):
    t = copy.deepcopy(cfg.template)
    t.contact_cone = abi.CONE_ELLIPTIC
    for profile in t.profiles:
        profile["law"] = abi.LAW_MUJOCO
    return t, {}


def servo_driven(cfg):
    """Position servos on every joint, ranges around the nominal pose on two of three, dry friction on every second."""
    t, g, E = copy.deepcopy(cfg.template), np.random.default_rng(23), cfg.env_count
    t.drive_rows, t.drive_mode = True, abi.DRIVE_PD_POSITION
    for l, link in enumerate(t.links):
        if link["joint_type"] != abi.JOINT_REVOLUTE:
            continue
        if l % 3 != 0:
            link["lower"], link["upper"] = float(cfg.nominal_q[l]) - 0.4, float(cfg.nominal_q[l]) + 0.5
        link["frictionloss"] = 0.15 if l % 2 == 0 else 0.0
    nl = t.link_count
    uploads = dict(drive_target=cfg.nominal_q + g.normal(0.0, 0.2, (E, nl)), drive_stiffness=np.tile(g.uniform(20.0, 80.0, nl), (E, 1)),
                   drive_damping=np.tile(g.uniform(0.5, 3.0, nl), (E, 1)), drive_force_limit=np.tile(g.uniform(15.0, 40.0, nl), (E, 1)))
    return t, {name: values.astype(np.float32) for name, values in uploads.items()}


@pytest.mark.parametrize("index,E,variant,before,spread", [
    (5, 4096, None, 0.887, 0.0063),              # 0.881: a wide block's forces and link motions as differences of running sums
    (3, 8192, elliptic, 0.9967, 0.0003),         # 0.9970: heads added in tiles at 36 coordinates
    (3, 16384, servo_driven, 0.9859, 0.0023),    # 0.9868: unit heads read together, contact heads without a question a head
])
def test_sums_in_another_order_end_as_near_the_double_solve(oracle_py, device, index, E, variant, before, spread):
    """The mean over the environments of the velocities' error, each taken as no more than the 95th percentile of the oracle's,
    as a share of the single-precision oracle's mean: `before` is what the loops that these sums replaced have on this batch,
    `spread` the standard deviation of new sums over old ones between batches of this size or half of it, and three
    of it are allowed.  (Over 32768 ropes and 65536 humanoids the new sums stand at 0.985, 1.0001 and 1.0004 of the old.)"""
    cfg = nk.synthetic.config(index, E)
    template, uploads = variant(cfg) if variant else (cfg.template, {})
    desc, state = abi.world_desc(E, cfg.dt, vel_iters=cfg.vel_iters), cfg.state()

    def stepped(w):
        w.set_state(state)
        for name, values in uploads.items():
            w.upload(name, values)
        w.step()
        if isinstance(w, nk.World):
            w.synchronize()
        out = w.download("link_velocity").astype(np.float64).reshape(E, -1), w.download("contact_count")
        assert not w.download("env_status").any()
        w.close()
        return out

    got, points = stepped(nk.World(device, template, desc))
    single, _ = stepped(oracle_py.OracleWorld(template, desc, threads=16))
    double, expect = stepped(oracle_py.OracleWorld(template, desc, threads=16, double=True))
    same = points == expect
    assert same.mean() > 0.99
    scale = np.maximum(np.linalg.norm(double, axis=1), 1e-2)
    device_error, oracle_error = (np.linalg.norm(v - double, axis=1)[same] / scale[same] for v in (got, single))
    cap = np.quantile(oracle_error, 0.95)
    share = np.minimum(device_error, cap).mean() / np.minimum(oracle_error, cap).mean()
    print(f"mean error {np.minimum(device_error, cap).mean():.3e}, {share:.4f} of the oracle's")
    assert share <= before + 3.0 * spread
