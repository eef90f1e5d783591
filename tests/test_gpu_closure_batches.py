"""The training step at batches around the gradient sum's 32 workgroups in
flight, and the weights it packs itself against a full repack."""
import numpy as np
import pytest

import ibgpu
import oracle_ffi as O

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def eng():
    mesh = ibgpu.Mesh(ibgpu.tiny_case())
    e = ibgpu.Engine(mesh, mode="mixed", turbulence=True)
    e.set_state(mesh.init_state())
    e.set_nut(np.full(mesh.ncells, mesh.phys[0].nut_inf))
    e.TimeMarching(0, 16)
    return e


def params(seed):
    prm = np.random.default_rng(seed).normal(0.0, 0.2, 4801 + 34).astype(np.float32)
    prm[4801:] = [0.0] * 8 + [1.0] * 8 + [-30.0] * 8 + [30.0] * 8 + [0.0, 1.0]
    return prm


@pytest.mark.parametrize("n", [1, 64 * 31, 64 * 32, 64 * 33 + 5, 64 * 64 + 1])
def test_gradient_of_many_workgroups(eng, n):
    eng.closure_init(1 << 12)
    prm = params(n)
    eng.closure_set_params(prm)
    rng = np.random.default_rng(n)
    x, z = rng.normal(size=(n, 8)).astype(np.float32), rng.normal(size=n).astype(np.float32)
    g, loss = eng.closure_grad(x, z)
    c, lc = O.mlp_grad(prm, x, z)
    # the mirror rounds to bf16 at the same points; the FP32 sums differ in
    # order, and a bf16 rounding they flip is 2^-9 of its value
    assert loss == pytest.approx(lc, rel=1e-4)
    assert np.linalg.norm(g - c) < 1e-3 * np.linalg.norm(c)


@pytest.mark.parametrize("batch", [64, 64 * 33])
def test_training_packs_its_weights(eng, batch):
    eng.closure_init(1 << 14)
    eng.closure_sample(0.9, 3)
    eng.closure_fit_stats(0.0)
    eng.closure_train(3, batch=batch, lr=1e-2, seed=4)
    x = np.random.default_rng(1).normal(size=(500, 8)).astype(np.float32)
    z0 = eng.closure_infer(x)
    g0, _ = eng.closure_grad(x, z0 + 1.0)
    eng.closure_set_params(eng.closure_params())     # repacks every layout
    z1 = eng.closure_infer(x)
    g1, _ = eng.closure_grad(x, z1 + 1.0)
    assert np.array_equal(z0, z1) and np.array_equal(g0, g1)
