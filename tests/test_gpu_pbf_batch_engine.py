"""The batched PBF engine (phx_pbf_batch_*): every pass of a substep is one
launch over all scenes, and with static boxes a captured substep is
replayed. Each scene's state equals its own PBF solver's bit for bit (and
the FP32 oracle's for the smallest scene), with graph replay and with eager
launches, over several calls with other work and synchronizations between
the replays; a scene with a moving box turns the replay off and still
matches."""
import numpy as np
import pytest
import torch

import oracle
from physica_amd import scenes
from physica_amd.batch import PbfBatch
from physica_amd.particle import ExecutionMode, PBF
from helpers import bits_equal, pbf_setup

pytestmark = pytest.mark.gpu

ITERATIONS = 3


def small_batch(count=5, moving=False):
    batch = [sc for sc in scenes.batched_pbf_scenes() if sc.count < 30_000][:count]
    if moving:
        b = batch[1].domain.boundary
        b.velocity = (0.05, 0.0, -0.02)
    return batch


def lone_states(batch, steps, device, iterations=ITERATIONS):
    """Each scene on its own PBF solver for `steps` steps."""
    out = []
    for sc in batch:
        solver, state, nxt, control, params, cache = pbf_setup(
            sc, device, PBF.Configuration(pressure_iterations=iterations), ExecutionMode.forward)
        states = [state, nxt]
        for k in range(steps):
            solver.forward_step(states[k % 2], control, params, states[(k + 1) % 2], cache)
        final = states[steps % 2]
        out.append((final.particles.positions.numpy(), final.particles.velocities.numpy()))
    torch.cuda.synchronize()
    return out


def batch_engine(batch, device, use_graph, iterations=ITERATIONS):
    engine = PbfBatch([sc.domain for sc in batch], PBF.Configuration(pressure_iterations=iterations),
                      use_graph=use_graph, device=device)
    state, control, params = engine.allocate_state(), engine.allocate_control(), engine.allocate_parameters()
    engine.upload(batch, state, params)
    return engine, state, control, params


def split(engine, state):
    x = state.particles.positions.numpy()
    v = state.particles.velocities.numpy()
    return [(x[:, engine.scene_slice(k)], v[:, engine.scene_slice(k)]) for k in range(engine.scene_count)]


def test_batch_offsets_and_launches(gpu_device):
    batch = small_batch()
    engine, state, control, params = batch_engine(batch, gpu_device, True)
    assert engine.offsets == list(np.cumsum([0] + [sc.count for sc in batch]))
    engine.run(state, control, params, 1)
    # counts fill, key, 3 scan kernels, scatter, rank, big-cell sort, gather,
    # 2 flag fills, the cell-bound fill, mask, 2 per iteration, vorticity,
    # normal, XSPH
    assert engine.kernels_per_step == 9 + 3 + 1 + 2 * ITERATIONS + 3
    assert state.particles.step_index == 1


@pytest.mark.parametrize("use_graph", [True, False])
def test_batch_equals_lone_solvers_over_replays(gpu_device, use_graph):
    print(f"pbf batch engine graph={use_graph}", flush=True)
    batch = small_batch()
    engine, state, control, params = batch_engine(batch, gpu_device, use_graph)
    done = 0
    for calls, steps in enumerate((3, 1, 4)):
        engine.run(state, control, params, steps)
        done += steps
        # eager work of the program between the replays, then a synchronize
        scratch = torch.randn(1 << 20, device=gpu_device)
        (scratch * 2.0).sum().item()
        torch.cuda.synchronize()
        assert state.particles.step_index == done
        expected = lone_states(batch, done, gpu_device)
        for k, ((x, v), (ex, ev)) in enumerate(zip(split(engine, state), expected)):
            assert bits_equal(x, ex), (calls, k)
            assert bits_equal(v, ev), (calls, k)


def test_batch_matches_the_oracle_and_a_moving_box(gpu_device):
    batch = small_batch(count=3, moving=True)
    engine, state, control, params = batch_engine(batch, gpu_device, True)
    engine.run(state, control, params, 2)
    torch.cuda.synchronize()
    expected = lone_states(batch, 2, gpu_device)
    got = split(engine, state)
    for k in range(len(batch)):
        assert bits_equal(got[k][0], expected[k][0]), k
        assert bits_equal(got[k][1], expected[k][1]), k
    smallest = min(range(len(batch)), key=lambda k: batch[k].count)
    sc = batch[smallest]
    d = oracle.make_domain(sc.domain)
    x, v = sc.positions, sc.velocities
    for step in range(2):
        r = oracle.pbf_step(d, step, x, v, np.zeros_like(x), sc.parameters, ITERATIONS)
        x, v = r["positions"], r["velocities"]
    assert bits_equal(got[smallest][0], x)
    assert bits_equal(got[smallest][1], v)


def test_batch_refuses_mixed_support_radii(gpu_device):
    batch = small_batch(count=2)
    batch[1].domain.support_radius = 0.05
    with pytest.raises(RuntimeError, match="support radius"):
        PbfBatch([sc.domain for sc in batch], PBF.Configuration(pressure_iterations=ITERATIONS), device=gpu_device)


@pytest.mark.parametrize("use_graph", [True, False])
@pytest.mark.parametrize("shapes", [((8, 8, 8), (9, 9, 9)), ((16, 16, 16), (10, 10, 10)), ((16, 16, 16),)])
def test_batch_without_pressure_iterations(gpu_device, shapes, use_graph):
    """0 iterations: the velocities come from the batch's reconstruction pass.
    Its blocks of 256 particles number 5, 20 and 16: fewer than the XCDs, not a
    multiple of them, and a multiple."""
    batch = [scenes.pbf_dam_break(shape=shape, seed=k) for k, shape in enumerate(shapes)]
    for k, sc in enumerate(batch):
        sc.velocities = np.random.default_rng(k).normal(0.0, 0.5, sc.positions.shape).astype(np.float32)
        sc.parameters["xsph_viscosity"][:] = 0.01
        sc.parameters["vorticity_confinement"][:] = 0.5
    engine, state, control, params = batch_engine(batch, gpu_device, use_graph, iterations=0)
    engine.run(state, control, params, 2)
    torch.cuda.synchronize()
    for (x, v), (lx, lv) in zip(split(engine, state), lone_states(batch, 2, gpu_device, iterations=0)):
        assert bits_equal(x, lx)
        assert bits_equal(v, lv)
