"""Ops dispatched and planned through the backend's function tables on views that a host has bound by field name."""
import ctypes as C

import numpy as np
import pytest

from conftest import nk
from test_gpu_chain import chain
from test_phi_views import view_fields

abi = nk.abi
pytestmark = pytest.mark.gpu
AHEAD = ("SnapshotStepVelocity", "FkWorldPoses", "ApplyDrives", "ArticulationDynamics", "IntegrateVelocity", "SyncLinkBodyPose", "BuildAabbs", "LbvhBuild",
         "LbvhQueryPairs", "NarrowphasePrimitives", "AssembleRows", "ContactWarmStart")
LEFT = ("lambda", "qdot", "link_velocity", "env_status", "vbd_velocity_sweep_count", "solver_residual")


class SolveParams(C.Structure):
    """BlockDescentSolveParams (src/phi/op_schema.hpp:596-640)."""
    _fields_ = [("dt", C.c_float)] + [(n, C.c_uint32) for n in (
        "iterations", "env_count", "rows_per_env", "total_particle_count", "total_body_count", "total_grid_count", "articulation_count", "max_dof",
        "base_link_count", "contact_rows_per_env", "contact_slots_per_env", "distinct_owner_rows_per_env", "joint_limit_rows_per_env")] + [
        ("incidence_per_env", C.c_uint64), ("measure_contact_residual", C.c_uint32), ("workspace_words", C.c_uint64), ("vertex_blocks", C.c_uint32 * 10),
        ("vertices_and_grids", C.c_uint32 * 8), ("clear_failure_diagnostics", C.c_uint32), ("substep_index", C.c_uint32), ("position_iterations", C.c_uint32),
        ("position_beta", C.c_float), ("position_slop", C.c_float), ("position_max_velocity", C.c_float), ("velocity_tolerance", C.c_float),
        ("trace_sweeps", C.c_uint32), ("telemetry", C.c_uint32), ("contact_anchors", C.c_uint32)]


def plain(name, text):
    """A parameter struct of four-byte members: `dt`s and `gravity` are floats."""
    kinds = {"dt": C.c_float, "gravity": C.c_float * 3}
    return type(name, (C.Structure,), {"_fields_": [(n, kinds.get(n, C.c_uint32)) for n in text.split()]})


PARAMS = {  # src/phi/op_schema.hpp:79-440
    "FkWorldPoses": plain("FkWorldPosesParams", "articulation_count total_link_count articulations_per_env selected_env_count"),
    "ApplyDrives": plain("ApplyDrivesParams", "dt total_link_count defer_velocity_damping mode links_per_env bodies_per_env articulation_count gravity"),
    "ArticulationDynamics": plain("ArticulationDynamicsParams", "dt max_dof integrate_velocity fold_drive_damping reuse_mass gravity articulation_count "
                                  "total_link_count apply_link_wrench max_links links_per_env bodies_per_env"),
    "IntegrateVelocity": plain("IntegrateVelocityParams", "dt gravity total_link_count articulation_count total_body_count clear_body_forces"),
    "IntegratePosition": plain("IntegratePositionParams", "dt total_link_count articulation_count total_body_count pos_pass env_count mimic_couplings"),
    "FkLinkVelocities": plain("FkLinkVelocitiesParams", "articulation_count total_link_count"),
    "SyncLinkBodyPose": plain("SyncLinkBodyPoseParams", "family env_count links_per_env bodies_per_env selected_env_count"),
    "BlockDescentSolve": SolveParams,
}


class OpCall(C.Structure):
    _fields_ = [("op", C.c_uint16), ("params", C.c_void_p)]


def table(handle, count):
    return C.cast(C.cast(handle, C.POINTER(C.c_void_p))[0], C.POINTER(C.c_void_p * count)).contents


class Host:
    """A backend of its own on the device, and the two views over memory that worlds hold (the first that has a field's)."""

    def __init__(self, worlds, counts):
        L = nk.lib()
        L.nuka_hip_model_view_bytes.restype = L.nuka_hip_data_view_bytes.restype = C.c_size_t
        self.model, self.data = [(C.c_char * size)() for size in (L.nuka_hip_model_view_bytes(), L.nuka_hip_data_view_bytes())]
        names = [f.name for f in view_fields()]
        self.bind(names, [1] * len(names))
        self.words = (C.c_uint64 * (len(self.data) // 8)).from_buffer(self.data)
        self.unnamed = [i for i, word in enumerate(self.words) if word == 0]   # places of the data view that no field stands for
        fields = [(f.name, worlds[f.owner if f.name in ROOMY else 0]._field(f.name.decode())[1].device_ptr) for f in view_fields()]
        self.bind(*zip(*fields))
        for name, value in counts.items():
            assert L.nuka_hip_model_view_set_count(self.model, name.encode(), value) == 0
        L.nuka_hip_register_backend_entry.restype = C.c_void_p
        entry = L.nuka_hip_register_backend_entry()
        handle = C.CFUNCTYPE(C.c_void_p, C.c_void_p, C.c_size_t)(table(entry, 4)[2])(entry, 0)
        self.backend = C.CFUNCTYPE(C.c_void_p, C.c_void_p, C.c_char_p)(table(handle, 6)[2])(handle, None)
        self.ops = table(self.backend, 15)

    def bind(self, names, pointers):
        nk.lib().nuka_hip_bind_views((C.c_char_p * len(names))(*names), (C.c_void_p * len(names))(*pointers), len(names), self.model, self.data, None, 0)

    def run(self, calls, planned):
        """(op, its parameters) in turn, or as one plan."""
        made = (OpCall * len(calls))(*[OpCall(nk.lib().nuka_hip_op_from_name(op.encode()), C.addressof(params)) for op, params in calls])
        views = [self.backend, C.addressof(self.model), C.addressof(self.data)]
        if planned:
            plan = C.CFUNCTYPE(C.c_void_p, C.c_void_p, C.c_void_p, C.c_void_p, C.c_void_p, C.c_int, C.c_void_p)(self.ops[4])(*views, C.addressof(made), len(calls), None)
            assert plan and C.CFUNCTYPE(C.c_uint8, C.c_void_p, C.c_void_p, C.c_void_p)(self.ops[5])(self.backend, plan, None) == 0
        else:
            for call in made:
                assert C.CFUNCTYPE(C.c_uint8, C.c_void_p, C.c_void_p, C.c_void_p, C.c_void_p)(self.ops[2])(*views, C.addressof(call)) == 0
        assert C.CFUNCTYPE(C.c_uint8, C.c_void_p, C.c_void_p)(self.ops[3])(self.backend, None) == 0
        if planned:
            C.CFUNCTYPE(None, C.c_void_p, C.c_void_p)(self.ops[6])(self.backend, plan)

    def close(self):
        C.CFUNCTYPE(None, C.c_void_p)(self.ops[1])(self.backend)


ROOMY = (b"m", b"m_factor", b"articulation_bias", b"articulation_qdd")   # by the coordinates of the view, not of the template


@pytest.mark.parametrize("planned", [False, True])
def test_what_no_field_stands_for_is_not_read_from_a_hosts_storage(device, planned):
    """A solve of more environments than the machine holds blocks, where a world's own launches take them from a queue: a pointer a
    host's storage holds in an unnamed place is left alone, and the solve is the world's."""
    E = 2784
    cfg = nk.synthetic.config(2, 96)
    for link in cfg.template.links:
        if link["joint_type"] == abi.JOINT_REVOLUTE:
            link["frictionloss"] = 0.1
    desc = abi.world_desc(E, cfg.dt, vel_iters=cfg.vel_iters, pos_iters=0xFFFFFFFF, velocity_tolerance=1e-5)   # no position pass
    state = {name: np.ascontiguousarray(np.asarray(v)[np.arange(E) % 96]) for name, v in cfg.state().items()}
    own, seam = nk.World(device, cfg.template, desc), nk.World(device, cfg.template, desc)
    for w in (own, seam):
        w.set_state(state)
        for op in AHEAD:
            w.op(op)
    own.op("BlockDescentSolve")
    own.synchronize()
    seam.upload("reset_env_ids", np.full(E, 0xABCD, np.uint32))
    seam.synchronize()

    info = seam.info
    frictions = info.links_per_env   # a dry-friction row a link, behind the contacts'
    assert E > 256 * info.solver_blocks_per_cu * 4 // 3   # (the queue's)
    contact_rows = info.rows_per_env - frictions
    host = Host((seam, seam), dict(
        links_per_env=info.links_per_env, bodies_per_env=info.bodies_per_env, dof=info.dof, max_dof=info.max_dof, contact_slots=info.contact_slots_per_env,
        rows_per_env=info.rows_per_env, contact_rows_per_env=contact_rows, floating_root=1, max_points_per_slot=1, joint_friction_rows=frictions))
    for at in host.unnamed:
        host.words[at] = seam._field("reset_env_ids")[1].device_ptr
    host.run([("BlockDescentSolve", SolveParams(
        dt=cfg.dt, iterations=cfg.vel_iters, env_count=E, rows_per_env=info.rows_per_env, total_body_count=E * info.bodies_per_env, articulation_count=E,
        max_dof=info.max_dof, base_link_count=info.links_per_env, contact_rows_per_env=contact_rows, contact_slots_per_env=info.contact_slots_per_env,
        velocity_tolerance=1e-5))], planned)
    host.close()
    assert (seam.download("reset_env_ids") == 0xABCD).all()
    assert (own.download("vbd_velocity_sweep_count") > 0).any()
    for name in LEFT:
        assert np.array_equal(own.download(name).view(np.uint8), seam.download(name).view(np.uint8)), name
    own.close()
    seam.close()


CHAIN_FIELDS = ("m", "m_factor", "articulation_bias", "articulation_qdd", "qdot", "qddot", "q", "link_velocity", "link_acceleration", "link_pose", "body_pose", "link_wrench")


@pytest.mark.parametrize("kinds,wide", [("RPFRR", 4), ("RPFRR", 7), ("PR", 8)])
@pytest.mark.parametrize("velocity,fold,pseudo,wrench", [(1, 0, 0, 1), (1, 1, 1, 0), (0, 1, 0, 1), (0, 0, 1, 0)])
@pytest.mark.parametrize("known", [1, 0])
def test_a_chains_plan_on_a_hosts_views(device, kinds, wide, velocity, fold, pseudo, wrench, known):
    """What no world asks for: matrices wider than the coordinates, velocities left alone, damping of the drives folded into the mass,
    pseudo-velocities.  A plan of a chain that the host names as one is a lane an environment, within single precision's rounding of
    the ops one by one (1e-5 of a field's norm, as test_gpu_chain.py has it); one that it does not is the ops', bit for bit."""
    E, dt, links = 70, 1.0 / 240.0, len(kinds)
    g = np.random.default_rng(10 * links + wide)
    t = chain(links, [dict(R=abi.JOINT_REVOLUTE, P=abi.JOINT_PRISMATIC, F=abi.JOINT_FIXED)[k] for k in kinds], g)
    moving = np.array([k != "F" for k in kinds])
    dof = int(moving.sum())
    state = {name: (g.normal(0.0, sigma, (E, links)) * moving).astype(np.float32) for name, sigma in (
        ("q", 1.0), ("qdot", 1.0), ("tau", 2.0), ("qdot_pseudo", 0.3), ("joint_gravity_force", 1.0))}
    state["drive_dissipation"] = g.uniform(0.1, 2.0, (E, links)).astype(np.float32)
    state["link_wrench"] = (g.normal(0.0, 1.0, (E, links, 6)) * (g.random((E, links, 1)) < 0.3)).astype(np.float32)
    base = np.zeros((E, 7), np.float32)
    base[:, 3] = 1.0
    everything = dict(articulation_count=E, total_link_count=E * links)
    down = dict(dt=dt, gravity=(C.c_float * 3)(0.5, -0.3, -9.81))
    calls = [
        ("FkWorldPoses", dict(everything, articulations_per_env=1)),
        ("ApplyDrives", dict(everything, **down, defer_velocity_damping=fold, mode=abi.DRIVE_TORQUE, links_per_env=links, bodies_per_env=links)),
        ("ArticulationDynamics", dict(everything, **down, max_dof=wide, integrate_velocity=velocity, fold_drive_damping=fold, apply_link_wrench=wrench, max_links=links,
                                      links_per_env=links, bodies_per_env=links)),
        ("IntegrateVelocity", dict(everything, **down, total_body_count=0)),
        ("IntegratePosition", dict(everything, dt=dt, pos_pass=pseudo, env_count=E)),
        ("FkWorldPoses", dict(everything, articulations_per_env=1)),
        ("FkLinkVelocities", everything),
        ("SyncLinkBodyPose", dict(env_count=E, links_per_env=links, bodies_per_env=links)),
    ]
    calls = [(op, PARAMS[op](**members)) for op, members in calls]
    out = []
    for planned in (False, True):
        own, roomy = nk.World(device, t, abi.world_desc(E, dt)), nk.World(device, chain(8, (abi.JOINT_REVOLUTE,), np.random.default_rng(0)), abi.world_desc(E, dt))
        own.set_state(dict(state, base_pose=base, root_twist=np.zeros((E, 6), np.float32)))
        for name in ("qdot_pseudo", "joint_gravity_force", "drive_dissipation", "link_wrench"):
            own.upload(name, state[name])
        for name in ROOMY:
            roomy.upload(name.decode(), np.full_like(roomy.download(name.decode()), 7.0))
        own.synchronize()
        info = own.info
        host = Host((own, roomy), dict(links_per_env=links, bodies_per_env=links, dof=dof, max_dof=wide, max_depth=links - 1, serial_chain=known,
                                       drive_mode=abi.DRIVE_TORQUE, sweep_passes=links))
        host.run(calls, planned)
        host.close()
        out.append({name: (roomy if name.encode() in ROOMY else own).download(name).astype(np.float64) for name in CHAIN_FIELDS})
        own.close()
        roomy.close()
    ops, plan = out
    assert info.dof == dof and np.abs(ops["articulation_qdd"][:E * wide]).max() > 0.1
    differs = False
    for name in CHAIN_FIELDS:
        if not known:
            assert np.array_equal(plan[name], ops[name]), name
        # (the words behind the view's matrices are not its own)
        assert np.array_equal(plan[name] == 7.0, ops[name] == 7.0) and np.linalg.norm(plan[name] - ops[name]) <= 1e-5 * np.linalg.norm(ops[name]), name
        differs = differs or not np.array_equal(plan[name], ops[name])
    assert differs == bool(known)
