"""FP64 kernels at the ends of their inputs' ranges, against the oracle: fluid
at rest without a Mach cut-off (a root of zero), an infinite Reynolds number
and walls so far away that the square of their distance overflows (infinite
divisors)."""
import numpy as np
import pytest

import ibgpu
import oracle_ffi
from test_gpu_parity import cols, perturbed_state

pytestmark = pytest.mark.gpu


def close(g, c):
    """Fifty roundings of terms that cancel by up to 10 within a column."""
    assert np.isfinite(c).all() and np.isfinite(g).all()
    assert (np.abs(g - c) <= 50 * 10 * 2.2e-16 * np.abs(c).max(0)).all()


@pytest.mark.parametrize("dim", [2, 3])
def test_fluid_at_rest_without_a_mach_cut_off(dim):
    mesh = ibgpu.Mesh(ibgpu.tiny_case() if dim == 2 else ibgpu.tiny3d_case())
    mesh.phys[0].Ma = 0.0
    fv = mesh.init_state()
    assert (fv[:, 2:4] == 0.0).all()
    eng = ibgpu.Engine(mesh, mode="fp64")
    eng.set_state(fv)
    c = oracle_ffi.Oracle(mesh, oracle_ffi.cfg(temporal_refine=0)).face_flux(fv, 0)
    close(eng.faceflux()[:, cols(mesh)], c[:, cols(mesh)])


@pytest.mark.parametrize("dim", [2, 3])
def test_infinite_reynolds_number(dim):
    mesh = ibgpu.Mesh(ibgpu.tiny_case() if dim == 2 else ibgpu.tiny3d_case())
    mesh.phys[0].Re = np.inf
    fv = perturbed_state(mesh)
    eng = ibgpu.Engine(mesh, mode="fp64")
    eng.set_state(fv)
    k = [1, 2, 3, 4] if dim == 3 else [1, 2, 4]
    c = oracle_ffi.Oracle(mesh, oracle_ffi.cfg(temporal_refine=0)).viscous_flux(fv, 0)[:, k]
    g = eng.vsflux()[:, k]
    assert (c[:, :-1] == 0.0).all() and (np.abs(g[:, :-1]) < 1e-250).all()
    close(g[:, -1:], c[:, -1:])


@pytest.mark.parametrize("dim", [2, 3])
def test_source_with_walls_far_away(dim):
    mesh = ibgpu.Mesh(ibgpu.tiny_case(Re=2000.0) if dim == 2 else ibgpu.tiny3d_case())
    r = np.random.default_rng(2)
    far = r.choice([0.0, 1e100, 1e160, 1e250, 1e308, np.inf], mesh.ncells)
    sd = np.where((far > 0.0) & (mesh.signdis > 0.0), far, mesh.signdis)
    mesh = oracle_ffi.PatchedMesh(mesh, signdis=sd)
    fv, nut = perturbed_state(mesh), mesh.phys[0].nut_inf * (0.5 + r.random(mesh.ncells))
    orc = oracle_ffi.Oracle(mesh, oracle_ffi.cfg(nstage=1, temporal_refine=0))
    _, mf = orc.viscous_flux_sa(fv, nut, 0)
    c = orc.mut_source(fv, nut, mf, 0)
    eng = ibgpu.Engine(mesh, mode="fp64", nstage=1, turbulence=True, temporal_refine=False)
    eng.set_state(fv)
    eng.set_nut(nut)
    eng.ComptViscousStress(0)
    eng.Stage(0, 0)
    used = (mesh.kind == 0) & (mesh.ibidx < 0) & (mesh.signdis > 0)
    assert (sd[used] > 1e150).any()
    close(eng.nut_source()[used, None], c[used, None])
