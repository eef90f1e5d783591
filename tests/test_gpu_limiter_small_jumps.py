"""FP64 limiters at differences down to the end of the FP64 range.

In a uniform stream along x the cross velocities start at exactly zero and the
front of a disturbance decays from cell to cell through every magnitude, past
the ones whose products and square sums are denormal or zero.  The slope there
is the one of a scaled-up flow: the momentum flux along a cross velocity
through the faces normal to another axis is linear in it.
"""
import numpy as np
import pytest

import ibgpu
import oracle_ffi

pytestmark = pytest.mark.gpu

MAGNITUDES = [1.0, 1e-150, 5e-155, 1e-157, 1e-160, 1e-161, 1e-180, 1e-250, 1e-290]


@pytest.fixture(scope="module")
def meshes():
    return {2: ibgpu.Mesh(ibgpu.tiny_case()), 3: ibgpu.Mesh(ibgpu.tiny3d_case())}


def uniform_with(mesh, comp, field):
    """The freestream with `field` as velocity component comp (2: v, 3: w)."""
    fv = mesh.init_state()
    fv[:, comp] = field
    P = mesh.phys[0]
    fv[:, 6] = P.Cv * fv[:, 5] + 0.5 * (fv[:, 1:4] ** 2).sum(1)
    return fv


@pytest.mark.parametrize("limiter", [0, 1])
@pytest.mark.parametrize("dim,comp", [(2, 2), (3, 2), (3, 3)])
def test_slope_of_small_differences(meshes, dim, comp, limiter):
    mesh = meshes[dim]
    r = np.random.default_rng(7)
    # steps of either sign between the cells, mostly growing along the axes
    field = mesh.centers @ np.array([1.0, 0.7, 0.4]) + 0.2 * r.random(mesh.ncells)
    field /= np.abs(field).max()
    eng = ibgpu.Engine(mesh, mode="fp64", limiter=limiter)
    orc = oracle_ffi.Oracle(mesh, oracle_ffi.cfg(temporal_refine=0, limiter=limiter))
    cross = mesh.face_dir != comp - 1
    for m in MAGNITUDES:
        fv = uniform_with(mesh, comp, 0.02 * m * field)
        eng.set_state(fv)
        g, c = eng.faceflux(), orc.face_flux(fv, 0)
        assert np.isfinite(g).all() and np.isfinite(c).all(), m
        g, c = g[cross, comp], c[cross, comp]
        # about fifty roundings of terms no larger than the largest flux (the
        # smallest area x velocity, 1e-290 x 1e-5, is still a normal number)
        assert np.abs(c).max() > 0.0
        assert (np.abs(g - c) <= 50 * 2.3e-16 * np.abs(c).max()).all(), m
    eng.close()


@pytest.mark.parametrize("name,subcycle,steps", [("config1", True, 60), ("config2", False, 30), ("tiny3d", True, 40)])
def test_van_albada_march_from_the_uniform_stream(name, subcycle, steps):
    """The default start: the disturbance of the section spreads into exactly
    zero cross velocities."""
    spec = {"config1": lambda: ibgpu.config1(levels=4, base=64), "config2": lambda: ibgpu.config2(levels=5, base=100),
            "tiny3d": ibgpu.tiny3d_case}[name]()
    mesh = ibgpu.Mesh(spec)
    fv = mesh.init_state()
    assert (fv[mesh.kind == 0, 2:4] == 0.0).all()
    orc = oracle_ffi.Oracle(mesh, oracle_ffi.cfg(nstage=3, dt_var_step=1 << (mesh.nlevels - 1) if subcycle else 1,
                                                 temporal_refine=int(subcycle), limiter=1))
    cpu, dt = fv.copy(), np.array([mesh.phys[0].dt_init])
    for ts in range(steps):
        assert orc.step(cpu, dt, ts)[0] == 0
    eng = ibgpu.Engine(mesh, mode="fp64", nstage=3, limiter=1, temporal_refine=subcycle)
    eng.set_state(fv)
    eng.TimeMarching(0, steps, use_graph=True)
    gpu = eng.get_state()
    eng.close()
    assert np.isfinite(gpu).all()
    # three stages a step of some fifty roundings (2.2e-16) each, relative to the norm
    assert np.linalg.norm(gpu[:, :5] - cpu[:, :5]) <= 3 * steps * 50 * 2.2e-16 * np.linalg.norm(cpu[:, :5])
