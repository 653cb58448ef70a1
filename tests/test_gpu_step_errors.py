"""What a failed step reports."""
import pytest

from conftest import nk
from test_gpu_head_capacity import crowded

pytestmark = pytest.mark.gpu
abi = nk.abi


@pytest.mark.parametrize("graph", [False, True])
def test_a_step_names_the_op_that_refused(device, graph):
    """A world of more contact slots than the row assembly's LDS takes (236): the ops before it, of which several share a
    launch, run, and the report names the assembly."""
    t, state = crowded(32, 2 * 240, 0.0, 2, seed=5)
    world = nk.World(device, t, abi.world_desc(2, 1.0 / 240.0, vel_iters=8, contact_margin=0.1))
    assert world.info.contact_slots_per_env == 240
    world.set_state(state)
    with pytest.raises(nk.NukaError) as err:
        world.set_execution_mode(graph)      # captures the plan
        world.step()
    assert err.value.code == abi.RESULT_INVALID_ARG
    info = world.execution_info()
    assert nk.lib().nuka_hip_op_name(info.failed_op).decode() == "AssembleRows"
    if not graph:
        assert info.message.decode() == "step failed in op AssembleRows"
    world.close()
