"""The solve of small blocks four environments a wavefront (batches from 8192 on): the batch's edges, more heads than a pass
takes, articulated blocks and single-axis heads, against the kernel that gives an environment a wavefront."""
import numpy as np
import pytest

from conftest import nk, per_env_error
from rigid import body_field, box_template
from test_gpu_parity import bar, one_ulp_sensitivity
from test_gpu_rigid import seeded_boxes
from trees import tree_case

pytestmark = pytest.mark.gpu
abi = nk.abi
STATE = ("qdot", "link_velocity", "lambda")


def repeated(values, count):
    values = np.asarray(values)
    return np.concatenate([values] * (count // len(values) + 1))[:count]


def copies_alike(big, name, E, count):
    """The batch repeats E environments: every copy holds the first one's bits."""
    batch = big.download(name).reshape(count, -1)
    assert np.array_equal(batch, repeated(batch[:E], count)), name
    return batch[:E]


# a last wavefront of one, two and three environments, and batches with and without environments that go alone; under the
# pyramidal cone the last batch that does not go four a wavefront and the first ones that do
@pytest.mark.parametrize("count", [8193, 8194, 8195, 12287, 12288, 12289, 12290, 12291, 24576, 24577])
@pytest.mark.parametrize("law", ["native", "pyramidal"])
def test_free_boxes_four_a_wavefront(device, count, law):
    E = 60
    t = box_template(half=(0.2, 0.15, 0.1), mass=3.0, diag=(0.03, 0.04, 0.05), mu=0.6)
    if law == "pyramidal":   # sixteen heads, on one axis each
        for profile in t.profiles:
            profile["law"] = abi.LAW_MUJOCO
        t.contact_cone = abi.CONE_PYRAMIDAL
    pose, v, w = seeded_boxes(E, 21)
    after = {}
    for envs in (E, count):
        world = nk.World(device, t, abi.world_desc(envs, 1.0 / 240.0, vel_iters=8, pos_iters=4, contact_margin=0.02))
        world.upload("base_pose", repeated(pose, envs))
        world.upload("body_linear_velocity", repeated(body_field(t, v), envs))
        world.upload("body_angular_velocity", repeated(body_field(t, w), envs))
        world.step(3); world.synchronize()
        names = ("base_pose", "body_linear_velocity", "body_angular_velocity", "lambda", "env_status", "vbd_velocity_sweep_count")
        after[envs] = {name: copies_alike(world, name, E, envs) for name in names}
        assert (world.download("contact_count") > 0).mean() >= 0.4
        world.close()
    for name, value in after[E].items():
        if law == "native" or value.dtype != np.float32:   # four heads: the same bits
            assert np.array_equal(value, after[count][name]), name
        else:   # the same sums in another grouping; three steps
            assert per_env_error(value, after[count][name], E, floor=1e-2).max() <= 3e-4, name


@pytest.mark.parametrize("dof,floating", [(4, False), (7, False), (8, True)])
def test_small_trees_four_a_wavefront(oracle_py, device, dof, floating):
    E, count = 48, 8192 + 31
    tree, desc, state = tree_case(oracle_py, dof, floating, True, seed=5 * dof + 1, E=E)
    small = nk.World(device, tree.template, desc)
    small.set_state(state)
    big = nk.World(device, tree.template, abi.world_desc(count, 1.0 / 240.0, vel_iters=8, contact_margin=0.1))
    big.set_state({k: repeated(v, count) for k, v in state.items()})
    for world in (small, big):
        assert world.dof == dof
        world.step(); world.synchronize()
    assert (small.download("contact_count") > 0).mean() >= 0.4, "the case must exercise the contact solve"
    sens = one_ulp_sensitivity(oracle_py, tree.template, desc, state)
    assert np.array_equal(copies_alike(big, "env_status", E, count).ravel(), small.download("env_status").ravel())
    for name in STATE:
        error = per_env_error(copies_alike(big, name, E, count), small.download(name), E).max()
        assert error <= bar(sens, "lambda" if name == "lambda" else "velocity"), (name, error)
    small.close(); big.close()


@pytest.mark.parametrize("count,packed", [(8192, False), (12287, False), (12288, True)])
def test_boxes_under_the_pyramidal_cone_go_four_a_wavefront_in_larger_batches(device, count, packed):
    """Six of the wavefronts of four fit a compute unit; they pay from 12288 environments on."""
    t = box_template(half=(0.2, 0.15, 0.1), mass=3.0, diag=(0.03, 0.04, 0.05), mu=0.6)
    for profile in t.profiles:
        profile["law"] = abi.LAW_MUJOCO
    t.contact_cone = abi.CONE_PYRAMIDAL
    world = nk.World(device, t, abi.world_desc(count, 1.0 / 240.0, vel_iters=8, contact_margin=0.02))
    assert (world.info.solver_blocks_per_cu == 6) == packed
    world.close()
