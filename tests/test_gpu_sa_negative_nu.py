"""FP64 SA source where the working variable is negative (set by the caller or
extrapolated; a march clips it at zero): r = nu / (S~ kappa^2 d^2 Re) is capped
at 10 from above only, so a weak vorticity takes it to -1e2 .. -1e9 and further,
where g^6 leaves the FP32 and then the FP64 range."""
import numpy as np
import pytest

import ibgpu
import oracle_ffi
from test_gpu_parity import perturbed_state

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("amp", [0.05, 1e-3, 1e-6, 1e-10])
@pytest.mark.parametrize("dim", [2, 3])
def test_source_of_a_negative_working_variable(dim, amp):
    mesh = ibgpu.Mesh(ibgpu.tiny_case(Re=2000.0) if dim == 2 else ibgpu.tiny3d_case())
    fv = perturbed_state(mesh, amp=amp)
    r = np.random.default_rng(3)
    nut = mesh.phys[0].nut_inf * r.choice([1.0, -1.0, -0.1, -3.0], mesh.ncells) * (0.5 + r.random(mesh.ncells))
    orc = oracle_ffi.Oracle(mesh, oracle_ffi.cfg(nstage=1, temporal_refine=0))
    _, mf = orc.viscous_flux_sa(fv, nut, 0)
    c = orc.mut_source(fv, nut, mf, 0)
    eng = ibgpu.Engine(mesh, mode="fp64", nstage=1, turbulence=True, temporal_refine=False)
    eng.set_state(fv)
    eng.set_nut(nut)
    eng.ComptViscousStress(0)
    eng.Stage(0, 0)
    g = eng.nut_source()
    used = (mesh.kind == 0) & (mesh.ibidx < 0) & (mesh.signdis > 0)
    g, c = g[used], c[used]
    assert np.isfinite(c).all() and np.isfinite(g).all()
    # some fifty roundings of terms that cancel by up to 1e3
    assert (np.abs(g - c) <= 1e3 * 50 * 2.2e-16 * (np.abs(c) + np.median(np.abs(c)))).all()
