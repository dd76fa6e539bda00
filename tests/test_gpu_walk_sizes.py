"""Forward steps bit-exact against the FP32 oracle (WCSPH up to the
platforms' powf) where the neighbour walks
change: particle counts around the sizes of waves and workgroups, particles
that move past every mask skin within a step, and neighbourhoods from empty
to more than twice a lattice's."""
import numpy as np
import pytest
import torch

import oracle
from physica_amd import scenes
from physica_amd.particle import DFSPH, PBF, ExecutionMode
from helpers import bits_equal, dfsph_setup, dfsph_state_numpy, pbf_setup, sph_setup

pytestmark = pytest.mark.gpu

COUNTS = (1, 15, 16, 17, 63, 64, 65, 255, 257, 1000, 5000)
# spacing of the particles over the scene's own (h is two of those): 0.79 gives up to 16 particles a cell and
# about 70 neighbours, 3 leaves a particle alone
SPREADS = (1.0, 0.79, 3.0)


def shrunk(sc, count, spread, seed, kick):
    """The scene's first `count` particles, their lattice scaled by `spread`
    inside the same box, with random velocities of `kick` supports a step."""
    rng = np.random.default_rng(seed)
    sc.positions = np.ascontiguousarray(sc.positions[:, :count] * np.float32(spread))
    reach = kick * sc.domain.support_radius / sc.domain.time_step
    sc.velocities = rng.normal(0.0, reach / 3.0, (3, count)).astype(np.float32)
    sc.parameters = {k: np.ascontiguousarray(v[:count]) for k, v in sc.parameters.items()}
    sc.parameters["masses"] = (sc.parameters["masses"] * rng.uniform(0.95, 1.05, count)).astype(np.float32)
    sc.domain.particle_count = count
    return sc


def lattice_for(count):
    side = 1
    while side ** 3 < count:
        side += 1
    return (side, side, side)


@pytest.mark.parametrize("count", COUNTS)
@pytest.mark.parametrize("spread", SPREADS)
@pytest.mark.parametrize("mode", [ExecutionMode.forward, ExecutionMode.differentiable])
def test_pbf(gpu_device, count, spread, mode):
    side = lattice_for(count)
    sc = shrunk(scenes.pbf_dam_break(shape=side, box=(2.0, 1.5, 1.5)), count, spread, count, 0.6)
    sc.parameters["xsph_viscosity"][:] = 0.01
    sc.parameters["vorticity_confinement"][:] = 0.5
    solver, state, nxt, control, params, cache = pbf_setup(sc, gpu_device, PBF.Configuration(3), mode)
    d = oracle.make_domain(sc.domain)
    x, v = sc.positions, sc.velocities
    for step in range(3):
        solver.forward_step(state, control, params, nxt, cache)
        torch.cuda.synchronize()
        exp = oracle.pbf_step(d, step, x, v, np.zeros_like(x), sc.parameters, 3)
        x, v = nxt.particles.positions.numpy(), nxt.particles.velocities.numpy()
        assert bits_equal(x, exp["positions"]), step
        assert bits_equal(v, exp["velocities"]), step
        state, nxt = nxt, state


@pytest.mark.parametrize("count", COUNTS)
@pytest.mark.parametrize("spread", SPREADS)
@pytest.mark.parametrize("mode,tolerance", [(ExecutionMode.forward, 0.0), (ExecutionMode.differentiable, 0.0),
                                            (ExecutionMode.forward, 1e-3)])
def test_dfsph(gpu_device, count, spread, mode, tolerance):
    side = lattice_for(count)
    sc = shrunk(scenes.dfsph_dam_break(shape=side, box=(0.4, 0.4, 0.4)), count, spread, count, 0.2)
    n = count
    cfg = DFSPH.Configuration(2, 3, density_error_tolerance=tolerance, max_iterations=5)
    solver, state, nxt, control, params, cache = dfsph_setup(sc, gpu_device, cfg, mode=mode)
    d = oracle.make_domain(sc.domain)
    x, v, u = sc.positions, sc.velocities, np.zeros_like(sc.positions)
    warm = (np.zeros(n, np.float32), np.zeros(n, np.float32))
    for step in range(3):
        solver.forward_step(state, control, params, nxt, cache)
        torch.cuda.synchronize()
        if tolerance > 0.0:
            exp = oracle.dfsph_step_tolerance(d, step, x, v, u, sc.parameters, warm[0], warm[1], tolerance, 5, True,
                                              "f32")
            assert solver.last_iterations() == exp["iterations"], step
        else:
            exp = oracle.dfsph_step(d, step, x, v, u, sc.parameters, warm[0], warm[1], 2, 3)
        got = dfsph_state_numpy(nxt)
        for name, value in got.items():
            assert bits_equal(value, exp[name]), (step, name)
        x, v = got["positions"], got["velocities"]
        warm = (got["warm_divergence_pressure"], got["warm_density_pressure"])
        state, nxt = nxt, state


@pytest.mark.parametrize("count", COUNTS)
@pytest.mark.parametrize("spread", SPREADS)
@pytest.mark.parametrize("method", ["iisph", "pcisph", "wcsph"])
def test_sph_methods(gpu_device, count, spread, method):
    side = lattice_for(count)
    sc = shrunk(scenes.two_cubes(method, shape=side, box=(4.0, 4.0, 2.0), spacing=0.05), count, spread, count, 0.2)
    if method == "wcsph":
        sc.parameters["tait_exponent"][:] = 1.0
        sc.parameters["viscosities"][:] = 0.05
        sc.parameters["surface_tensions"][:] = 0.5
    else:
        sc.parameters["viscosities"][:] = 0.01
    solver, state, nxt, control, params, cache = sph_setup(sc, gpu_device, method, pressure_iterations=3)
    d = oracle.make_domain(sc.domain)
    x, v, u = sc.positions, sc.velocities, np.zeros_like(sc.positions)
    for step in range(3):
        solver.forward_step(state, control, params, nxt, cache)
        torch.cuda.synchronize()
        if method == "wcsph":
            exp = oracle.wcsph_step(d, step, x, v, u, sc.parameters)
        else:
            exp = oracle.pressure_solver_step(d, step, x, v, u, sc.parameters, method, 3)
        x, v = nxt.particles.positions.numpy(), nxt.particles.velocities.numpy()
        if method == "wcsph":
            # the platforms' powf(r, 1) differ by an ulp of the density ratio r here and there: by dp = rho0 c^2
            # 2^-23 r, and sum m |grad W| / rho <= 12 / h, so |dv| <= dt c^2 2^-22 r 12 / h, plus the rounding of v
            ratio = float(exp["densities"].max()) / 1000.0
            bound = sc.domain.time_step * 7.0 * 2.0**-22 * ratio * 12.0 / sc.domain.support_radius
            assert np.abs(v - exp["velocities"]).max() <= bound + 2.0**-23 * np.abs(v).max(), step
        else:
            assert bits_equal(x, exp["positions"]), step
            assert bits_equal(v, exp["velocities"]), step
        state, nxt = nxt, state


@pytest.mark.parametrize("shape", [(30, 20, 30), (60, 30, 60)])
def test_pbf_cells_with_many_boundary_samples(gpu_device, shape):
    """More than 16 boundary samples in a cell, in a scene whose passes run
    their workgroups in order (18,000 particles) and in one that starts the
    workgroups with crowded particles first (108,000)."""
    sc = scenes.pbf_dam_break(shape=shape)
    s = 2.0 * float(sc.domain.particle_radius)
    x = np.arange(30) * s / 3.0
    gx, gz = np.meshgrid(x + sc.positions[0].min(), x + sc.positions[2].min(), indexing="ij")
    pos = np.stack([gx.ravel(), np.full(gx.size, -0.5 * s), gz.ravel()]).astype(np.float32)
    vel = np.zeros_like(pos)
    vol = np.full(pos.shape[1], s ** 3 / 9.0, np.float32)
    sc.domain.boundary_particles = [(tuple(p), (0.0, 0.0, 0.0), float(w)) for p, w in zip(pos.T, vol)]
    solver, state, nxt, control, params, cache = pbf_setup(sc, gpu_device, PBF.Configuration(2))
    solver.forward_step(state, control, params, nxt, cache)
    torch.cuda.synchronize()
    d = oracle.make_domain(sc.domain, (pos, vel, vol))
    exp = oracle.pbf_step(d, 0, sc.positions, sc.velocities, np.zeros_like(sc.positions), sc.parameters, 2)
    assert bits_equal(nxt.particles.positions.numpy(), exp["positions"])
    assert bits_equal(nxt.particles.velocities.numpy(), exp["velocities"])
