"""Block tiles (16 x 16 squares, in 3D 8 x 8 x 4 boxes of cells processed
without face lists, used with the default tile of 256 cells) against general
tiles over the same cells (a tile of 128 cells has none): the same state
after a sub-cycling period, bit for bit in the mixed mode, to rounding in
FP64."""
import numpy as np
import pytest

import ibgpu

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def meshes():
    # ragged bases: blocks, general runs between them and partial tiles on
    # every level; spans of 3, 6 and 12 cells
    return {2: ibgpu.Mesh(ibgpu.config2(levels=5, base=90)), 3: ibgpu.Mesh(ibgpu.config3(levels=4, base=42, nz=3))}


def flow(mesh):
    x, d = mesh.centers, np.clip(mesh.signdis, 0.0, 10.0)
    fv = mesh.init_state()
    fv[:, 0] *= 1.0 + 0.01 * np.sin(3.0 * x[:, 0] + x[:, 1])
    fv[:, 1] *= 1.0 - 0.8 * np.exp(-d / 0.05)
    fv[:, 2] += 0.02 * np.cos(2.0 * x[:, 1] - x[:, 0])
    if mesh.dim == 3:
        fv[:, 3] += 0.01 * np.sin(60.0 * x[:, 2] + x[:, 0])
    fv[:, 4] *= 1.0 + 0.01 * np.cos(x[:, 0] * 2.0)
    nut = mesh.phys[0].nut_inf * (1.0 - 0.9 * np.exp(-d / 0.1))
    return fv, nut


CASES = [
    ("fp64", "laminar", {}), ("fp64", "sa", {}), ("fp64", "sa", dict(nstage=4, limiter=1)),
    ("fp64", "laminar", dict(viscous=False)), ("fp64", "laminar", dict(temporal_refine=False, reflux=True)),
    ("mixed", "laminar", {}), ("mixed", "sa", {}), ("mixed", "sa", dict(nstage=4, limiter=1)),
    ("mixed", "sa", dict(nstage=1)), ("mixed", "laminar", dict(viscous=False)),
    ("mixed", "learned", dict(nstage=4)), ("mixed", "learned", dict(schedule=1)),
    ("mixed", "sa", dict(schedule=1)), ("mixed", "sa", dict(temporal_refine=False, reflux=True)),
]


@pytest.mark.parametrize("dim", [2, 3])
@pytest.mark.parametrize("mode,closure,opt", CASES)
def test_block_tiles_equal_general_tiles(meshes, dim, mode, closure, opt):
    mesh = meshes[dim]
    fv, nut = flow(mesh)
    steps = 1 << (mesh.nlevels - 1) if opt.get("temporal_refine", True) else 2
    if opt.get("nstage", 3) == 1:
        steps = 1
    got = {}
    for tile in (0, 128):
        eng = ibgpu.Engine(mesh, mode=mode, tile=tile, turbulence=closure != "laminar",
                           **dict(dict(nstage=3), **opt))
        if closure == "learned":
            prm = np.random.default_rng(5).normal(0.0, 0.1, 4801 + 34).astype(np.float32)
            prm[4801:] = [0.0] * 8 + [3.0] * 8 + [-30.0] * 8 + [30.0] * 8 + [0.02, 0.02]
            eng.closure_init(1024)
            eng.closure_set_params(prm)
            eng.closure_enable(True)
        eng.set_state(fv)
        if closure != "laminar":
            eng.set_nut(nut)
        eng.TimeMarching(0, steps, use_graph=steps > 1)
        linf, l2 = eng.ResinDomain()
        got[tile] = (eng.get_state(), eng.get_nut() if closure != "laminar" else np.zeros(1), linf, l2,
                     eng.bench_stage(0, 0, 1)[1:])
        eng.close()
    a, b = got[0], got[128]
    # the squares list no faces: the default tiling really has block tiles
    assert a[4][0] == b[4][0] and a[4][1] < 0.6 * b[4][1]
    if mode == "mixed":
        assert np.array_equal(a[0], b[0]) and np.array_equal(a[1], b[1])
        assert np.array_equal(a[2], b[2])
    else:
        # the direction known at compile time may fuse other products: a few
        # roundings (2.2e-16) a stage, 64 stages at most
        for k in (0, 1):
            assert np.linalg.norm(a[k] - b[k]) <= 64 * 2.2e-16 * np.linalg.norm(b[k])
        assert np.allclose(a[2], b[2], rtol=1e-9, atol=1e-300)
    assert np.allclose(a[3], b[3], rtol=1e-9, atol=1e-300)   # sums in another order
