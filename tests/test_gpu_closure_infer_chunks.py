"""Inference in chunks of 16384 rows through two pinned buffers: row counts
around the chunk, a later larger call after a small one, and the entry point
without allocations as the second route."""
import numpy as np
import pytest

import ibgpu
import oracle_ffi as O

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def eng():
    e = ibgpu.Engine(ibgpu.Mesh(ibgpu.tiny_case()), mode="mixed", turbulence=True)
    e.closure_init(1024)
    prm = np.random.default_rng(3).normal(0.0, 0.2, 4801 + 34).astype(np.float32)
    prm[4801:] = [0.0] * 8 + [1.0] * 8 + [-30.0] * 8 + [30.0] * 8 + [0.5, 2.0]
    e.closure_set_params(prm)
    return e, prm


@pytest.mark.parametrize("n", [1, 255, 1025, 16383, 16384, 16385, 2 * 16384, 3 * 16384 + 77])
def test_chunked_inference(eng, n):
    e, prm = eng
    x = np.random.default_rng(n).normal(size=(n, 8)).astype(np.float32)
    z = e.closure_infer(x)
    assert np.array_equal(z, e.closure_infer(x))
    if n <= 65536:
        assert np.array_equal(z, e.closure_infer_noalloc(x))
    c = O.mlp_forward(prm, x)
    # the mirror rounds to bf16 at the same points
    assert np.linalg.norm(z - c) < 1e-3 * np.linalg.norm(c)
