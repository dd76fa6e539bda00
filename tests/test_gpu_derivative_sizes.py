"""Derivative passes against the FP64 oracle where their neighbour walks
change: particle counts around the sizes of waves and workgroups and on both
sides of the count from which a particle gets fewer lanes."""
import numpy as np
import pytest
import torch

import oracle
import test_gpu_dfsph_derivatives as dfsph
from physica_amd import scenes
from physica_amd.particle import PBF, ExecutionMode
from physica_amd.rollout import PbfRollout
from helpers import bits_equal, pbf_setup

pytestmark = pytest.mark.gpu

DFSPH_LIMIT = 40000  # 16 lanes a particle up to here
PBF_FIELDS = ("relaxation", "xsph_viscosity", "vorticity_confinement")


def pbf_scene(count, seed):
    side = 1
    while side ** 3 < count:
        side += 1
    sc = scenes.pbf_dam_break(shape=(side, side, side), box=(4.0, 3.0, 3.0))
    rng = np.random.default_rng(seed)
    jitter = rng.uniform(-0.2, 0.2, (3, count)) * sc.domain.support_radius / 2.0
    sc.positions = (sc.positions[:, :count] + jitter).astype(np.float32)
    sc.velocities = rng.normal(0.0, 0.3, (3, count)).astype(np.float32)
    sc.parameters = {k: np.ascontiguousarray(v[:count]) for k, v in sc.parameters.items()}
    sc.parameters["masses"] = (sc.parameters["masses"] * rng.uniform(0.95, 1.05, count)).astype(np.float32)
    sc.parameters["xsph_viscosity"][:] = 0.01
    sc.parameters["vorticity_confinement"][:] = 0.2
    sc.domain.particle_count = count
    return sc


def adjoints(solver, prev_a, ctl_a, par_a):
    got = {"positions": prev_a.particles.positions.numpy(), "velocities": prev_a.particles.velocities.numpy(),
           "controls": ctl_a.external_accelerations.numpy(), "masses": par_a.particles.masses.cpu().numpy(),
           "rest_densities": par_a.particles.rest_densities.cpu().numpy()}
    for k in PBF_FIELDS:
        got[k] = getattr(par_a, k).cpu().numpy()
    return got


@pytest.mark.parametrize("count", [1, 15, 17, 63, 65, 257, 1000, 20000, 20001])
@pytest.mark.parametrize("iterations", [0, 1, 3])
def test_pbf_vjp(gpu_device, count, iterations):
    sc = pbf_scene(count, count + iterations)
    solver, state, nxt, control, params, cache = pbf_setup(sc, gpu_device, PBF.Configuration(iterations),
                                                           ExecutionMode.differentiable)
    solver.forward_step(state, control, params, nxt, cache)
    rng = np.random.default_rng(3)
    wx, wv = rng.normal(0, 1, (3, count)), rng.normal(0, 1, (3, count))
    next_a, prev_a = solver.allocate_state_adjoint(), solver.allocate_state_adjoint()
    next_a.particles.positions.upload(wx)
    next_a.particles.velocities.upload(wv)
    ctl_a, par_a = solver.allocate_control_adjoint(), solver.allocate_parameter_adjoint()
    solver.vjp_step(state, control, params, nxt, cache, next_a, prev_a, ctl_a, par_a)
    torch.cuda.synchronize()
    exp = oracle.pbf_vjp(oracle.make_domain(sc.domain), 0, sc.positions, sc.velocities, np.zeros_like(sc.positions),
                         sc.parameters, wx, wv, iterations)
    for k, value in adjoints(solver, prev_a, ctl_a, par_a).items():
        # sums of some 100 terms in another order: 100 x 2^-53 of the terms' magnitudes per pass, some ten passes,
        # and cancellation to about a thousandth of them at the largest adjoint
        scale = max(np.abs(exp[k]).max(), 1e-300)
        assert np.abs(value - exp[k]).max() / scale < 1e-10, k


def test_rollout_records_over_its_caches(gpu_device):
    """Three passes through one rollout: each gives the gradient of its own
    forward pass, and a final state that the caller holds is left alone."""
    sc = pbf_scene(1000, 5)
    solver, state, _, control, params, _ = pbf_setup(sc, gpu_device, PBF.Configuration(2),
                                                     ExecutionMode.differentiable)
    other = solver.allocate_state()
    solver.copy_state(state, other)
    other.particles.positions.x.add_(0.01)

    def run(rollout, start):
        final = rollout.forward(start, control, params)
        seed = solver.allocate_state_adjoint()
        seed.particles.positions.upload(np.ones((3, 1000)))
        initial, ctl, par = rollout.backward(seed)
        torch.cuda.synchronize()
        return final, adjoints(solver, initial, ctl, par)

    fresh = [run(PbfRollout(solver, 3), s) for s in (state, other, state)]
    rollout = PbfRollout(solver, 3)
    held = [run(rollout, s) for s in (state, other, state)]
    for (final, got), (expected_final, expected) in zip(held, fresh):
        assert bits_equal(final.particles.positions.numpy(), expected_final.particles.positions.numpy())
        for k in expected:
            assert np.array_equal(got[k], expected[k]), k
    rollout.release()
    final, got = run(rollout, other)
    assert all(np.array_equal(got[k], fresh[1][1][k]) for k in got)


def dfsph_case(count):
    """A lattice of `count` particles off the cell borders, swirling, with some
    moving further within the step than any mask skin."""
    side = 1
    while side ** 3 < count:
        side += 1
    sc = scenes.dfsph_dam_break(shape=(side, side, side), box=(0.8, 0.8, 0.8))
    rng = np.random.default_rng(count)
    h = sc.domain.support_radius
    jitter = rng.uniform(-0.1, 0.1, (3, count)) * h
    sc.positions = (0.95 * sc.positions[:, :count] + 0.1 + jitter).astype(np.float32)
    velocities = rng.normal(0.0, 0.05, (3, count))
    velocities[:, ::7] += 0.3 * h / sc.domain.time_step * rng.uniform(-1.0, 1.0, (3, velocities[:, ::7].shape[1]))
    sc.velocities = velocities.astype(np.float32)
    sc.parameters = {k: np.ascontiguousarray(v[:count]) for k, v in sc.parameters.items()}
    sc.parameters["masses"] = (sc.parameters["masses"] * rng.uniform(0.95, 1.05, count)).astype(np.float32)
    sc.parameters["viscosities"][:] = 0.01
    sc.domain.particle_count = count
    zeros = np.zeros(count, np.float32)
    return dfsph.Case(sc, oracle.make_domain(sc.domain), (zeros, zeros))


@pytest.mark.parametrize("count", [1, 15, 17, 63, 65, 257, 1000, DFSPH_LIMIT, DFSPH_LIMIT + 1])
def test_dfsph_derivatives(gpu_device, count):
    cs = dfsph_case(count)
    run = dfsph.recorded(cs, gpu_device, 1, 2, True)
    t, w = dfsph.directions(cs, np.random.default_rng(4))
    x, v, u, p, wd, we = dfsph.inputs(cs, "f32")
    got = dfsph.run_vjp(*run, w, gpu_device)
    exp = oracle.dfsph_vjp(cs.d, 0, x, v, u, p, wd, we, w, 1, 2, True, "f32")
    for k in dfsph.STATE + dfsph.PARAMS + dfsph.WARM:
        # as for PBF: FP64 sums in another order
        assert np.abs(got[k] - exp[k]).max() <= 1e-10 * max(np.abs(exp[k]).max(), 1e-300), k
    got = dfsph.run_jvp(*run, t, gpu_device)
    exp = oracle.dfsph_jvp(cs.d, 0, x, v, u, p, wd, we, t, 1, 2, True, "f32")
    for k in ("positions", "velocities") + dfsph.WARM:
        # the oracle's FP32 operations in its order; the platforms' functions differ by units of the last place
        assert np.abs(got[k] - exp[k]).max() <= 1e-6 * max(np.abs(exp[k]).max(), 1e-30), k
