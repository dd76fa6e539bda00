"""PBF::forward_step on the GPU vs the FP32 oracle: bit-exact with the
reference parameters; artificial pressure (powf) within a stated tolerance."""
import numpy as np
import pytest
import torch

import oracle
from physica_amd import scenes
from physica_amd.batch import PbfBatch
from physica_amd.particle import PBF
from helpers import bits_equal, max_rel, pbf_setup

pytestmark = pytest.mark.gpu


def gpu_step(solver, state, nxt, control, params, cache):
    solver.forward_step(state, control, params, nxt, cache)
    torch.cuda.synchronize()
    return nxt.particles.positions.numpy(), nxt.particles.velocities.numpy()


def test_dam_break_32k_bit_exact_rollout(gpu_device):
    """The 32,768-particle PBF dam break: 10 substeps, each bit-exact against the
    oracle fed the same input; cache fields bit-exact on the last step."""
    sc = scenes.pbf_dam_break()
    solver, state, nxt, control, params, cache = pbf_setup(sc, gpu_device)
    d = oracle.make_domain(sc.domain)
    x, v = sc.positions, sc.velocities
    for step in range(10):
        gx, gv = gpu_step(solver, state, nxt, control, params, cache)
        exp = oracle.pbf_step(d, step, x, v, np.zeros_like(x), sc.parameters, 4)
        assert bits_equal(gx, exp["positions"]), step
        assert bits_equal(gv, exp["velocities"]), step
        x, v = gx, gv
        solver.copy_state(nxt, state)
    rho, lam = cache.last_iteration()
    assert bits_equal(rho.cpu().numpy(), exp["densities"])
    assert bits_equal(lam.cpu().numpy(), exp["lambdas"])
    assert bits_equal(cache.predicted_positions().numpy(), exp["predicted_positions"])
    keys, idx, off = cache.neighborhood()
    ok, oi, oo = oracle.build_neighborhood(d, 10, exp["predicted_positions"])
    assert np.array_equal(idx.cpu().numpy().astype(np.uint32), oi)
    assert np.array_equal(off.cpu().numpy().astype(np.uint32), oo)


@pytest.mark.parametrize("iterations", [0, 1, 5])
def test_vorticity_and_xsph_bit_exact(gpu_device, iterations):
    sc = scenes.pbf_dam_break(shape=(16, 16, 16))
    n = sc.count
    rng = np.random.default_rng(3)
    sc.velocities = rng.normal(0, 0.5, size=(3, n)).astype(np.float32)
    sc.parameters["xsph_viscosity"] = rng.uniform(0, 0.05, n).astype(np.float32)
    sc.parameters["vorticity_confinement"] = rng.uniform(0, 0.5, n).astype(np.float32)
    solver, state, nxt, control, params, cache = pbf_setup(sc, gpu_device, PBF.Configuration(iterations))
    gx, gv = gpu_step(solver, state, nxt, control, params, cache)
    exp = oracle.pbf_step(oracle.make_domain(sc.domain), 0, sc.positions, sc.velocities, np.zeros((3, n)),
                          sc.parameters, iterations)
    assert bits_equal(gx, exp["positions"])
    assert bits_equal(gv, exp["velocities"])


def test_artificial_pressure_within_tolerance(gpu_device):
    """s_corr uses powf per pair; device and host powf may differ in the last
    ulp, so this case is held to 1e-5 relative rather than bit equality."""
    sc = scenes.pbf_dam_break(shape=(16, 16, 16))
    n = sc.count
    sc.parameters["artificial_pressure_strength"] = np.full(n, 1e-4, np.float32)
    solver, state, nxt, control, params, cache = pbf_setup(sc, gpu_device)
    gx, gv = gpu_step(solver, state, nxt, control, params, cache)
    exp = oracle.pbf_step(oracle.make_domain(sc.domain), 0, sc.positions, sc.velocities, np.zeros((3, n)),
                          sc.parameters, 4)
    motion = np.abs(exp["positions"] - sc.positions).max()
    assert np.abs(gx - exp["positions"]).max() <= 1e-5 * motion
    assert max_rel(gv, exp["velocities"]) <= 1e-5


@pytest.mark.parametrize("batched", [False, True])
def test_masses_outside_the_quick_division(gpu_device, batched):
    """Masses and rest densities whose quotients the pair terms cannot take
    from a reciprocal (the remainders underflow), then usual ones, then the
    first again: bit-exact steps, of a solver and of one batch's replays."""
    sc = scenes.pbf_dam_break(shape=(12, 12, 12))
    rng = np.random.default_rng(9)
    usual = dict(sc.parameters)
    tiny = dict(usual)
    tiny["masses"] = (rng.uniform(1.0, 2.0, sc.count) * 2.0**-118).astype(np.float32)
    tiny["rest_densities"] = np.full(sc.count, 1.37 * 2.0**-60, np.float32)
    tiny["relaxation"] = np.full(sc.count, 2.0**-34, np.float32)  # corrections of some 1e-3
    d = oracle.make_domain(sc.domain)
    u = np.zeros_like(sc.positions)
    engine = PbfBatch([sc.domain], PBF.Configuration(2), use_graph=True, device=gpu_device)
    state, control, params = engine.allocate_state(), engine.allocate_control(), engine.allocate_parameters()
    for parameters in (tiny, usual, tiny):
        sc.parameters = parameters
        exp = oracle.pbf_step(d, 0, sc.positions, sc.velocities, u, parameters, 2)
        free = oracle.pbf_step(d, 0, sc.positions, sc.velocities, u, parameters, 0)
        assert np.abs(exp["positions"] - free["positions"]).max() > 1e-4
        if batched:
            engine.upload([sc], state, params)  # into the arrays that the captured substep reads
            state.particles.step_index = 0
            engine.run(state, control, params, 1)
            torch.cuda.synchronize()
            gx, gv = state.particles.positions.numpy(), state.particles.velocities.numpy()
        else:
            gx, gv = gpu_step(*pbf_setup(sc, gpu_device, PBF.Configuration(2)))
        assert bits_equal(gx, exp["positions"])
        assert bits_equal(gv, exp["velocities"])


def test_masses_back_in_range(gpu_device):
    """One solver: a step with a mass outside the quick range, then one without."""
    sc = scenes.pbf_dam_break(shape=(8, 8, 8))
    solver, state, nxt, control, params, cache = pbf_setup(sc, gpu_device, PBF.Configuration(2))
    d = oracle.make_domain(sc.domain)
    for mass in (np.float32(2.0**-70), sc.parameters["masses"][7]):
        p = dict(sc.parameters)
        p["masses"] = p["masses"].copy()
        p["masses"][7] = mass
        params.particles.masses.copy_(torch.from_numpy(p["masses"]))
        exp = oracle.pbf_step(d, 0, sc.positions, sc.velocities, np.zeros_like(sc.positions), p, 2)
        state.particles.step_index = 0
        gx, gv = gpu_step(solver, state, nxt, control, params, cache)
        assert bits_equal(gx, exp["positions"])
        assert bits_equal(gv, exp["velocities"])
