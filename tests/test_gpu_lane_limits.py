"""Forward steps bit-exact against the FP32 oracle (WCSPH up to the platforms'
powf) on both sides of the particle counts where the passes change their lanes
per particle: 20,000 and 90,000 for the SPH methods (16, 4 and 1), 32,768 for
PBF (16 and 4). Velocities take particles past their mask skins, the first
step's displacements set the per-cell skins of the next ones, and clumps of
particles in single cells make crowded neighbourhoods; masses are unequal or
equal (candidates as position and pressure records). The counts end in part of
a workgroup."""
import numpy as np
import pytest
import torch

import oracle
from physica_amd import scenes
from physica_amd.particle import DFSPH, IISPH, PBF, SPH, ExecutionMode
from helpers import add_boundary_samples, bits_equal, dfsph_setup, dfsph_state_numpy, pbf_setup, sph_setup
from test_gpu_walk_sizes import lattice_for, shrunk

pytestmark = pytest.mark.gpu


def with_clumps(sc, seed, equal_masses=False, clumps=((3, 2, 4), 300), more=((8, 9, 7), 40)):
    """Moves random particles into two cells (300 and 40 of them)."""
    rng = np.random.default_rng(seed)
    h = sc.domain.support_radius
    moved = rng.permutation(sc.count)
    start = 0
    for cell, count in (clumps, more):
        lo = (np.array(cell, dtype=np.float64) + 0.05) * h
        chosen = moved[start:start + count]
        sc.positions[:, chosen] = (lo[:, None] + rng.uniform(0.0, 0.9 * h, (3, count))).astype(np.float32)
        start += count
    if equal_masses:
        sc.parameters["masses"][:] = sc.parameters["masses"][0]
    return sc


def dfsph_scene(count, equal_masses=False):
    side = lattice_for(count)
    sc = shrunk(scenes.dfsph_dam_break(shape=side, box=(0.6, 0.6, 0.6)), count, 1.0, count, 0.2)
    return with_clumps(sc, count, equal_masses)


def run_dfsph(sc, samples, device, tolerance, steps=3):
    n = sc.count
    cfg = DFSPH.Configuration(2, 2, density_error_tolerance=tolerance, max_iterations=3)
    solver, state, nxt, control, params, cache = dfsph_setup(sc, device, cfg)
    d = oracle.make_domain(sc.domain, samples)
    x, v, u = sc.positions, sc.velocities, np.zeros_like(sc.positions)
    warm = (np.zeros(n, np.float32), np.zeros(n, np.float32))
    for step in range(steps):
        solver.forward_step(state, control, params, nxt, cache)
        torch.cuda.synchronize()
        if tolerance > 0.0:
            exp = oracle.dfsph_step_tolerance(d, step, x, v, u, sc.parameters, warm[0], warm[1], tolerance, 3, True,
                                              "f32")
            assert solver.last_iterations() == exp["iterations"], step
        else:
            exp = oracle.dfsph_step(d, step, x, v, u, sc.parameters, warm[0], warm[1], 2, 2)
        got = dfsph_state_numpy(nxt)
        for name, value in got.items():
            assert bits_equal(value, exp[name]), (step, name)
        x, v = got["positions"], got["velocities"]
        warm = (got["warm_divergence_pressure"], got["warm_density_pressure"])
        state, nxt = nxt, state


@pytest.mark.parametrize("count", [20000, 20001, 90000, 90001])
@pytest.mark.parametrize("equal_masses,tolerance", [(False, 0.0), (True, 0.0), (False, 1e-3)])
def test_dfsph(gpu_device, count, equal_masses, tolerance):
    run_dfsph(dfsph_scene(count, equal_masses), None, gpu_device, tolerance)


@pytest.mark.parametrize("tolerance", [0.0, 1e-3])
def test_dfsph_with_samples(gpu_device, tolerance):
    sc = dfsph_scene(20001)
    run_dfsph(sc, add_boundary_samples(sc, moving=True), gpu_device, tolerance)


def sph_scene(method, count, equal_masses=False):
    side = lattice_for((count + 1) // 2)
    sc = scenes.two_cubes(method, shape=side, box=(4.0, 4.0, 3.0), spacing=0.05)
    sc = with_clumps(shrunk(sc, count, 1.0, count, 0.2), count, equal_masses)
    if method == "wcsph":
        sc.parameters["tait_exponent"][:] = 1.0
        sc.parameters["viscosities"][:] = 0.05
        sc.parameters["surface_tensions"][:] = 0.5
    else:
        sc.parameters["viscosities"][:] = 0.01
    return sc


def run_sph(sc, method, samples, device, tolerance=0.0, steps=3):
    solver, state, nxt, control, params, cache = sph_setup(sc, device, method, pressure_iterations=2)
    if tolerance > 0.0:
        solver = SPH(sc.domain, IISPH.Configuration(density_error_tolerance=tolerance, max_iterations=4), device=device)
        cache = solver.allocate_step_cache()
    d = oracle.make_domain(sc.domain, samples)
    x, v, u = sc.positions, sc.velocities, np.zeros_like(sc.positions)
    for step in range(steps):
        solver.forward_step(state, control, params, nxt, cache)
        torch.cuda.synchronize()
        if method == "wcsph":
            exp = oracle.wcsph_step(d, step, x, v, u, sc.parameters)
        elif tolerance > 0.0:
            exp = oracle.pressure_solver_step_tolerance(d, step, x, v, u, sc.parameters, method, tolerance, 4)
        else:
            exp = oracle.pressure_solver_step(d, step, x, v, u, sc.parameters, method, 2)
        x, v = nxt.particles.positions.numpy(), nxt.particles.velocities.numpy()
        if method == "wcsph":
            # the bound of test_gpu_walk_sizes.test_sph_methods: an ulp of the density ratio through powf(r, 1)
            ratio = float(exp["densities"].max()) / 1000.0
            bound = sc.domain.time_step * 7.0 * 2.0**-22 * ratio * 12.0 / sc.domain.support_radius
            assert np.abs(v - exp["velocities"]).max() <= bound + 2.0**-23 * np.abs(v).max(), step
        else:
            assert bits_equal(x, exp["positions"]), step
            assert bits_equal(v, exp["velocities"]), step
        state, nxt = nxt, state


@pytest.mark.parametrize("count", [20001, 90001])
@pytest.mark.parametrize("method,equal_masses,tolerance", [("iisph", False, 0.0), ("iisph", True, 0.0),
                                                           ("iisph", False, 1e-3), ("pcisph", False, 0.0)])
def test_pressure_solvers(gpu_device, method, count, equal_masses, tolerance):
    run_sph(sph_scene(method, count, equal_masses), method, None, gpu_device, tolerance)


def test_wcsph(gpu_device):
    run_sph(sph_scene("wcsph", 20001), "wcsph", None, gpu_device)


@pytest.mark.parametrize("method", ["iisph", "wcsph"])
def test_sph_with_samples(gpu_device, method):
    sc = sph_scene(method, 20001)
    if method == "wcsph":
        sc.parameters["boundary_surface_tension"][:] = 0.5
    run_sph(sc, method, add_boundary_samples(sc), gpu_device)


def run_pbf(sc, device, mode, steps):
    solver, state, nxt, control, params, cache = pbf_setup(sc, device, PBF.Configuration(2), mode)
    d = oracle.make_domain(sc.domain)
    x, v = sc.positions, sc.velocities
    for step in range(steps):
        solver.forward_step(state, control, params, nxt, cache)
        torch.cuda.synchronize()
        exp = oracle.pbf_step(d, step, x, v, np.zeros_like(x), sc.parameters, 2)
        x, v = nxt.particles.positions.numpy(), nxt.particles.velocities.numpy()
        assert bits_equal(x, exp["positions"]), step
        assert bits_equal(v, exp["velocities"]), step
        state, nxt = nxt, state


def pbf_scene(count, spread=1.0):
    side = lattice_for(count)
    sc = shrunk(scenes.pbf_dam_break(shape=side, box=(3.2, 2.4, 2.4)), count, spread, count, 0.6)
    sc.parameters["xsph_viscosity"][:] = 0.01
    sc.parameters["vorticity_confinement"][:] = 0.5
    return sc


@pytest.mark.parametrize("count", [32768, 32769])
@pytest.mark.parametrize("mode", [ExecutionMode.forward, ExecutionMode.differentiable])
def test_pbf(gpu_device, count, mode):
    run_pbf(with_clumps(pbf_scene(count), count), gpu_device, mode, steps=2)


def test_pbf_with_more_crowded_workgroups_than_are_served_early(gpu_device):
    """100,003 particles about 24 to a cell: nearly every one of the passes'
    1,563 workgroups is crowded, of which 512 are listed to start first."""
    sc = pbf_scene(100003, spread=0.7)
    cells = np.floor((sc.positions.astype(np.float64)) / sc.domain.support_radius).astype(np.int64)
    _, members = np.unique(cells, axis=1, return_counts=True)
    assert members[members > 16].sum() > 0.8 * sc.count
    run_pbf(sc, gpu_device, ExecutionMode.forward, steps=1)
