"""Ops dispatched and planned through the backend's function tables on views that a host has bound by field name."""
import ctypes as C

import numpy as np
import pytest

from conftest import nk
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


class OpCall(C.Structure):
    _fields_ = [("op", C.c_uint16), ("params", C.c_void_p)]


def table(handle, count):
    return C.cast(C.cast(handle, C.POINTER(C.c_void_p))[0], C.POINTER(C.c_void_p * count)).contents


def bound_views(world, counts):
    """The two views over a world's own memory, and where the data view has words that no field stands for."""
    L = nk.lib()
    L.nuka_hip_model_view_bytes.restype = L.nuka_hip_data_view_bytes.restype = C.c_size_t
    model, data = [(C.c_char * size)() for size in (L.nuka_hip_model_view_bytes(), L.nuka_hip_data_view_bytes())]
    names = [f.name for f in view_fields()]
    c_names = (C.c_char_p * len(names))(*names)
    L.nuka_hip_bind_views(c_names, (C.c_void_p * len(names))(*([1] * len(names))), len(names), model, data, None, 0)
    words = (C.c_uint64 * (len(data) // 8)).from_buffer(data)
    unnamed = [i for i, word in enumerate(words) if word == 0]
    pointers = [world._field(name.decode())[1].device_ptr for name in names]
    L.nuka_hip_bind_views(c_names, (C.c_void_p * len(names))(*pointers), len(names), model, data, None, 0)
    for name, value in counts.items():
        assert L.nuka_hip_model_view_set_count(model, name.encode(), value) == 0
    return model, data, words, unnamed


@pytest.mark.parametrize("planned", [False, True])
def test_what_no_field_stands_for_is_not_read_from_a_hosts_storage(device, planned):
    """A solve of more environments than the machine holds blocks, where a world's own launches take them from a queue: a pointer a
    host's storage holds in an unnamed place is left alone, and the solve is the world's."""
    E = 2304
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

    L, info = nk.lib(), seam.info
    frictions = info.links_per_env   # a dry-friction row a link, behind the contacts'
    assert E > 256 * info.solver_blocks_per_cu
    contact_rows = info.rows_per_env - frictions
    model, data, words, unnamed = bound_views(seam, dict(
        links_per_env=info.links_per_env, bodies_per_env=info.bodies_per_env, dof=info.dof, max_dof=info.max_dof, contact_slots=info.contact_slots_per_env,
        rows_per_env=info.rows_per_env, contact_rows_per_env=contact_rows, floating_root=1, max_points_per_slot=1, joint_friction_rows=frictions))
    for at in unnamed:
        words[at] = seam._field("reset_env_ids")[1].device_ptr
    params = SolveParams(dt=cfg.dt, iterations=cfg.vel_iters, env_count=E, rows_per_env=info.rows_per_env, total_body_count=E * info.bodies_per_env,
                         articulation_count=E, max_dof=info.max_dof, base_link_count=info.links_per_env, contact_rows_per_env=contact_rows,
                         contact_slots_per_env=info.contact_slots_per_env, velocity_tolerance=1e-5)
    call = OpCall(L.nuka_hip_op_from_name(b"BlockDescentSolve"), C.addressof(params))
    L.nuka_hip_register_backend_entry.restype = C.c_void_p
    entry = L.nuka_hip_register_backend_entry()
    handle = C.CFUNCTYPE(C.c_void_p, C.c_void_p, C.c_size_t)(table(entry, 4)[2])(entry, 0)
    backend = C.CFUNCTYPE(C.c_void_p, C.c_void_p, C.c_char_p)(table(handle, 6)[2])(handle, None)
    ops = table(backend, 15)
    two, three = C.CFUNCTYPE(C.c_uint8, C.c_void_p, C.c_void_p), C.CFUNCTYPE(C.c_uint8, C.c_void_p, C.c_void_p, C.c_void_p)
    if planned:
        plan = C.CFUNCTYPE(C.c_void_p, C.c_void_p, C.c_void_p, C.c_void_p, C.c_void_p, C.c_int, C.c_void_p)(ops[4])(
            backend, C.addressof(model), C.addressof(data), C.addressof(call), 1, None)
        assert plan and three(ops[5])(backend, plan, None) == 0
    else:
        assert C.CFUNCTYPE(C.c_uint8, C.c_void_p, C.c_void_p, C.c_void_p, C.c_void_p)(ops[2])(
            backend, C.addressof(model), C.addressof(data), C.addressof(call)) == 0
    assert two(ops[3])(backend, None) == 0
    if planned:
        C.CFUNCTYPE(None, C.c_void_p, C.c_void_p)(ops[6])(backend, plan)
    C.CFUNCTYPE(None, C.c_void_p)(ops[1])(backend)
    assert (seam.download("reset_env_ids") == 0xABCD).all()
    assert (own.download("vbd_velocity_sweep_count") > 0).any()
    for name in LEFT:
        assert np.array_equal(own.download(name).view(np.uint8), seam.download(name).view(np.uint8)), name
    own.close()
    seam.close()
