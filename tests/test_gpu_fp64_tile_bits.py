"""FP64: tile size and schedule change the launch shape only, also on meshes
most of whose cells lie in block tiles (which only a tile of 256 cells has):
the same bits from every tile size, from one workgroup per tile and from
persistent workgroups, so that an autotuned run does not depend on which
tile was the fastest."""
import numpy as np
import pytest

import ibgpu
from test_gpu_block_tiles import flow

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def meshes():
    # ragged bases: blocks, general runs between them and partial tiles on
    # every level
    return {2: ibgpu.Mesh(ibgpu.config2(levels=5, base=90)), 3: ibgpu.Mesh(ibgpu.config3(levels=4, base=42, nz=3))}


CASES = [
    ("laminar", {}), ("sa", {}), ("sa", dict(nstage=4, limiter=1)), ("laminar", dict(viscous=False)),
    ("sa", dict(temporal_refine=False)), ("laminar", dict(temporal_refine=False, reflux=True)), ("sa", dict(nstage=1)),
]


@pytest.mark.parametrize("dim", [2, 3])
@pytest.mark.parametrize("closure,opt", CASES)
def test_fp64_bits_do_not_depend_on_the_tile(meshes, dim, closure, opt):
    mesh = meshes[dim]
    fv, nut = flow(mesh)
    opt = dict(dict(nstage=3), **opt)
    steps = 1 if opt["nstage"] == 1 else 4
    ref = None
    for tile, schedule in ((128, 0), (0, 0), (0, 1), (64, 0), (192, 1)):
        eng = ibgpu.Engine(mesh, mode="fp64", tile=tile, schedule=schedule, turbulence=closure == "sa", **opt)
        eng.set_state(fv)
        if closure == "sa":
            eng.set_nut(nut)
        eng.TimeMarching(0, steps, use_graph=schedule == 1)
        got = [eng.get_state(), eng.ResinDomain()[0]] + ([eng.get_nut()] if closure == "sa" else [])
        cells, faces = eng.bench_stage(0, 0, 1)[1:]
        eng.close()
        if ref is None:
            ref, ref_faces = got, faces
            continue
        if tile == 0:   # the squares list no faces
            assert faces < 0.6 * ref_faces
        for x, y in zip(got, ref):
            assert np.array_equal(x, y), (tile, schedule)
