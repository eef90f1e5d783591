"""FP64 face flux where its limiter quotients degenerate: equal neighbours
(0/0), jumps whose ratio passes the reference's 1e10 guard with either sign,
and velocity jumps whose product underflows, against the oracle."""
import numpy as np
import pytest

import ibgpu
import oracle_ffi

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("limiter", [0, 1])
@pytest.mark.parametrize("dim", [2, 3])
def test_flux_of_degenerate_jumps(dim, limiter):
    mesh = ibgpu.Mesh(ibgpu.tiny_case() if dim == 2 else ibgpu.tiny3d_case())
    r = np.random.default_rng(11)
    n = mesh.ncells
    jump = lambda small: r.choice([0.0, 0.0, small, -small, 3e-2, -1e-2, 1e-5], n)
    fv = mesh.init_state()
    fv[:, 0] *= 1.0 + jump(1e-14)
    fv[:, 1] *= 1.0 + jump(1e-14)
    fv[:, 2] = jump(1e-180)
    if dim == 3:
        fv[:, 3] = jump(1e-300)
    fv[:, 4] *= 1.0 + jump(1e-13)
    P = mesh.phys[0]
    fv[:, 5] = fv[:, 4] / (fv[:, 0] * P.Rg)
    fv[:, 6] = P.Cv * fv[:, 5] + 0.5 * (fv[:, 1:4] ** 2).sum(1)
    eng = ibgpu.Engine(mesh, mode="fp64", limiter=limiter)
    eng.set_state(fv)
    g = eng.faceflux()
    c = oracle_ffi.Oracle(mesh, oracle_ffi.cfg(temporal_refine=0, limiter=limiter)).face_flux(fv, 0)
    assert np.isfinite(g).all() and np.isfinite(c).all()
    # about fifty roundings of terms no larger than a column's largest flux,
    # whose parts cancel by up to p / (roe u^2) ~ 10
    tol = 50 * 10 * 2.3e-16 * np.abs(c).max(0)
    assert (np.abs(g - c) <= tol).all()
