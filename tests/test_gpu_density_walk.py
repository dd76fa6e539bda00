"""The two-phase walk of the density primitives against the FP32 oracle where
it can go wrong: lists that fill up on the way, cells of one to hundreds of
particles, and values outside the support that are not finite."""
import numpy as np
import pytest
import torch

import oracle
from physica_amd import DeviceBoundary, build_neighborhood, density_forward, density_jvp, density_vjp
from physica_amd.particle import (ParticleParameterAdjoint, ParticleParameters, ParticleParameterTangent,
                                  VectorAdjointField, VectorField)
from test_gpu_neighborhood import boundary_samples, domain, with_boundary

pytestmark = pytest.mark.gpu


def same(a, b):
    """Equal bit for bit, any NaN equal to any other."""
    nan = np.isnan(a)
    return np.array_equal(nan, np.isnan(b)) and np.array_equal(a[~nan], b[~nan])


# per scene: particles in one spot of that radius (the support is 0.05), particles spread over the box
SCENES = {"list_just_full": (40, 0.005, 0), "list_over_by_one": (41, 0.005, 0), "two_lists": (83, 0.005, 500),
          "one_cell": (700, 0.01, 300), "alone": (1, 0.0, 0), "spread": (0, 0.0, 257)}


@pytest.mark.parametrize("scene", sorted(SCENES))
@pytest.mark.parametrize("pbf_kernel", [False, True])
@pytest.mark.parametrize("samples", [0, 400])
@pytest.mark.parametrize("special", [None, np.nan, np.inf])
def test_density_walk_equals_oracle(gpu_device, scene, pbf_kernel, samples, special):
    spot, radius, spread = SCENES[scene]
    n = spot + spread
    rng = np.random.default_rng(n + 2 * pbf_kernel + samples)
    x = np.concatenate([0.31 + rng.uniform(-radius, radius, (3, spot)),
                        rng.uniform(0.0, 0.6, (3, spread))], axis=1)[:, rng.permutation(n)].astype(np.float32)
    xt = rng.normal(size=(3, n)).astype(np.float32)
    m, r0 = rng.uniform(0.5, 1.5, n).astype(np.float32), rng.uniform(900, 1100, n).astype(np.float32)
    mt, rt = rng.normal(size=n).astype(np.float32), rng.normal(size=n).astype(np.float32)
    w = rng.normal(size=n)
    if special is not None:  # it reaches every particle of the 27 cells, as 0 times it is NaN
        m[n // 2] = special
        xt[1, n // 3] = special
    cfg, boundary, packed = domain(n), None, None
    if samples:
        packed = boundary_samples(rng, samples, moving=True)
        cfg = with_boundary(cfg, packed)
        boundary = DeviceBoundary(cfg, gpu_device)
    dev = lambda a, dt=torch.float32: torch.from_numpy(np.ascontiguousarray(a)).to(device=gpu_device, dtype=dt)  # noqa: E731
    xf, tf = VectorField.zeros(n, gpu_device), VectorField.zeros(n, gpu_device)
    xf.upload(x)
    tf.upload(xt)
    z, zd = torch.zeros(n, device=gpu_device), torch.zeros(n, device=gpu_device, dtype=torch.float64)
    params = ParticleParameters(dev(m), dev(r0), z, z)
    step, h = 2, cfg.support_radius
    nb = build_neighborhood(cfg, step, xf, gpu_device)
    rho, rho_t = torch.empty(n, device=gpu_device), torch.empty(n, device=gpu_device)
    density_forward(h, pbf_kernel, xf, xf, params, nb.view, rho, boundary, nb.boundary_time)
    density_jvp(h, pbf_kernel, xf, xf, tf, params, ParticleParameterTangent(dev(mt), dev(rt), z, z), nb.view, rho_t,
                boundary, nb.boundary_time)
    pos_a = VectorAdjointField(*(zd.clone() for _ in range(3)))
    par_a = ParticleParameterAdjoint(zd.clone(), zd.clone(), zd, zd)
    density_vjp(h, pbf_kernel, xf, xf, params, nb.view, dev(w, torch.float64), pos_a, par_a, boundary,
                nb.boundary_time)
    torch.cuda.synchronize()
    od = oracle.make_domain(cfg, packed) if samples else oracle.make_domain(cfg)
    assert same(rho.cpu().numpy(), oracle.density(od, step, pbf_kernel, x, x, m, r0))
    assert same(rho_t.cpu().numpy(), oracle.density_jvp(od, step, pbf_kernel, x, x, xt, m, mt, r0, rt))
    ea, em, er = oracle.density_vjp(od, step, pbf_kernel, x, x, m, r0, w)
    assert same(pos_a.numpy(), ea)
    assert same(par_a.masses.cpu().numpy(), em)
    assert same(par_a.rest_densities.cpu().numpy(), er)
