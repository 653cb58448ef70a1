"""Contact heads that act on nothing: rows between two sides that do not move are heads of the solve without a place among
its staged rows, whichever place among the heads they have."""
import numpy as np
import pytest

from conftest import make_pair, nk
from test_gpu_parity import ORACLE_OPS, ROW_WORDS, UPSTREAM, bar, one_ulp_sensitivity, scaled_errors, velocity_scale

pytestmark = pytest.mark.gpu
ACTIVE, BLOCK_TANGENT, STATIC = 1 << 0, 1 << 3, 3


# full blocks sum four heads a pass, the humanoid's reduced block three: `idle` leaves passes that are in part empty
@pytest.mark.parametrize("index,idle", [(2, (0,)), (2, (0, 1, 2)), (2, (1, 3)), (3, (0,)), (3, (0, 1)), (3, (2, 5, 7))])
def test_heads_without_a_moving_side_change_nothing_for_the_others(oracle_py, device, index, idle):
    E = 96
    cfg, oracle, world, state = make_pair(oracle_py, device, index, E)
    desc = nk.abi.world_desc(E, cfg.dt, vel_iters=cfg.vel_iters)
    sens = one_ulp_sensitivity(oracle_py, cfg.template, desc, state)
    for name in UPSTREAM:
        oracle.op(*ORACLE_OPS[name])
        world.op(name)
    world.synchronize()
    R = world.rows_per_env
    made = 0
    for w in (oracle, world):
        rows = w.download("urows")
        words = rows.view(np.uint32).reshape(E, R, ROW_WORDS)
        for e in range(E):
            flags = words[e, :, 0]
            heads = np.flatnonzero(((flags & ACTIVE) != 0) & ((flags & BLOCK_TANGENT) == 0))
            for h in idle:
                if h >= heads.size:
                    continue
                at = heads[h] + words[e, heads[h], 2] * np.arange(3)      # its normal row and, a stride apart, its tangents
                words[e, at, 10] = STATIC
                words[e, at, 18] = STATIC
                made += 1
        w.upload("urows", rows)
    assert made >= E                                    # both worlds, half of the environments at least
    scale = velocity_scale(world, oracle, E)
    oracle.op("block_descent_solve")
    world.op("BlockDescentSolve")
    world.synchronize()
    assert np.array_equal(world.download("env_status"), oracle.download("env_status"))
    error = scaled_errors(world.download("qdot_flat"), oracle.download("qdot_flat"), scale, E)
    print(f"config {index}, idle heads {idle}: velocities {error.max():.2e} from the oracle's")
    assert error.max() <= bar(sens, "velocity")
    world.close()
    oracle.close()
