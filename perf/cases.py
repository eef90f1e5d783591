"""Timed workloads of the residual engine: what its users have it do.

A run is a time march of a section (or a batch of sections) on its AMR level
set: the state goes in, the march runs from captured graphs or step by step,
and the state, the working variable, dt, the residual norms and the wall
force come out.  Beside the marches: the training of the learned closure on
rows sampled from a run, its inference over rows handed in by the host, and
the regrid of a moving section.

listed() names the workloads, draw() gives others of the same ranges,
prepare() builds what a program holds before the call (mesh, context,
initial state, weights), run() is one pass, work() the bytes and operations
a pass cannot do without, exact() the result in 64 bits where it has a
closed form.
"""
import dataclasses
import functools
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                                "immsered-boundary_amd"))

import ibgpu  # noqa: E402

# pitch and heave of the moving section: x0, y0, aoa0, amplitude (deg), omega, heave
MOTION = (0.0, 0.0, 0.0, 5.0, 0.2, 0.05)
NPARAM = 4801
# standardisation of the closure's eight features (ln|Omega|, vorticity share,
# ln d, ln chi, ln Re_d, roe, p/p_inf, ln nu): the spread over the fluid cells
FMEAN = (-3.0, 0.5, 0.0, 1.5, 8.0, 1.0, 1.0, 0.0)
FSTD = (4.0, 0.4, 1.5, 1.0, 3.0, 0.1, 0.1, 0.1)


def _march(name, **kw):
    c = dict(kind="march", dim=2, section="naca0012", base=64, levels=4, nz=1, sections=1, mode="fp64",
             closure="laminar", moving=False, stages=4, limiter=0, subcycle=True, reflux=False,
             steps=64, stepwise=False)
    c.update(kw)
    if name:
        c["name"] = name
    return c


def listed():
    return [
        # a small laminar case driven step by step from the host, as the C++
        # driver does: one step, then the residual norms, a few launches each
        _march("steps_small_laminar_fp64", stages=3, steps=16, stepwise=True),
        # a small SA case left to run: graph replay, a few tens of thousand cells
        _march("march_small_sa_mixed", base=96, levels=5, mode="mixed", closure="sa"),
        # mid-size laminar case without sub-cycling, van Albada, with the
        # coarse/fine flux balance: every level marched every step
        _march("march_mid_laminar_fp64_balanced", section="naca0015", base=100, levels=5, stages=3,
               limiter=1, subcycle=False, reflux=True, steps=32),
        # the moving NACA0015 section, 2.6M cells, re-tagged every step:
        # plain FP64, mixed precision, mixed with the learned closure
        _march("march_2d_moving_sa_fp64", section="naca0015", base=256, levels=6, closure="sa",
               moving=True, steps=128),
        _march("march_2d_moving_sa_mixed", section="naca0015", base=256, levels=6, mode="mixed",
               closure="sa", moving=True, steps=256),
        _march("march_2d_moving_learned", section="naca0015", base=256, levels=6, mode="mixed",
               closure="learned", moving=True, steps=256),
        # the quasi-span 3D section
        _march("march_3d_sa_fp64", dim=3, base=64, levels=5, nz=4, closure="sa", steps=32),
        _march("march_3d_sa_mixed", dim=3, base=64, levels=5, nz=4, mode="mixed", closure="sa", steps=64),
        # eight sections of uneven refinement in one launch sequence
        _march("ensemble_sa_mixed", section="ensemble", base=128, levels=6, sections=8, mode="mixed",
               closure="sa", steps=128),
        # the closure's training: Adam steps on batches of the sampled rows
        dict(name="closure_training", kind="train", base=100, levels=5, rows=1000000, batch=8192, steps=100),
        # inference over rows from the host: an odd number of rows
        dict(name="closure_inference", kind="infer", rows=100003),
        # the level set rebuilt at a new pose handed to the running context
        dict(name="regrid_moving_mixed", kind="regrid", base=128, levels=6, angle=0.05),
    ]


def draw(rng):
    def log_int(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    pick = rng.random()
    if pick < 0.12:
        return dict(kind="infer", rows=log_int(1, 1000000))
    if pick < 0.24:
        return dict(kind="train", base=log_int(64, 110), levels=5, rows=log_int(9000, 1000000),
                    batch=64 * log_int(8, 128), steps=log_int(10, 100))
    if pick < 0.30:
        return dict(kind="regrid", base=2 * log_int(56, 64), levels=6, angle=round(rng.uniform(0.01, 0.08), 4))
    mode = rng.choice(("fp64", "mixed"))
    closure = rng.choice(("laminar", "sa", "sa", "learned"))
    if closure == "learned":
        mode = "mixed"
    stages = rng.choice((3, 4))
    if pick < 0.48:
        return _march(None, dim=3, base=2 * log_int(18, 30), levels=rng.choice((4, 5)), nz=rng.choice((3, 4)),
                      mode=mode, closure=closure, stages=stages, steps=log_int(8, 32))
    if pick < 0.60:
        fine = rng.random() < 0.5
        return _march(None, section="ensemble", base=log_int(117, 128) if fine else log_int(64, 110),
                      levels=6 if fine else 5, sections=rng.randint(2, 6), mode=mode, closure=closure, stages=stages,
                      steps=log_int(16, 96))
    subcycle = rng.random() < 0.8
    levels = rng.choice((5, 6))
    section = rng.choice(("naca0012", "naca0015"))
    # the finest band of the larger section has to hold its wall cells
    lo = 64 if section == "naca0012" else (112 if levels == 6 else 68)
    return _march(None, section=section, base=log_int(lo, 230), levels=levels,
                  mode=mode, closure=closure, moving=subcycle and rng.random() < 0.5, stages=stages,
                  limiter=rng.choice((0, 0, 1)), subcycle=subcycle,
                  reflux=not subcycle and rng.random() < 0.5,
                  steps=log_int(16, 96) if subcycle else log_int(8, 32), stepwise=rng.random() < 0.2)


# ------------------------------------------------------------------ prepare
def _specs(section, dim, base, levels, nz, sections, aoa=None):
    if section == "ensemble":
        return ibgpu.ensemble_cases(n=sections, base=base, levels=levels)
    if dim == 3:
        return [ibgpu.config3(levels=levels, base=base, nz=nz)]
    spec = ibgpu.config2(levels=levels, base=base) if section == "naca0015" else ibgpu.config1(levels=levels, base=base)
    spec = dataclasses.replace(spec, inlet_nut="freestream")
    return [spec if aoa is None else dataclasses.replace(spec, aoa=aoa)]


@functools.lru_cache(maxsize=3)
def _mesh(section, dim, base, levels, nz, sections, aoa=None):
    # the level set does not depend on the seed: built once per process
    return ibgpu.Mesh(_specs(section, dim, base, levels, nz, sections, aoa))


def _mesh_of(case):
    return _mesh(case["section"], case["dim"], case["base"], case["levels"], case["nz"], case["sections"])


def _flow(mesh, seed):
    """A flow of the kind the march meets: the freestream with a slowed layer
    along the wall and a smooth disturbance of a percent, the working
    variable growing away from the wall."""
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    g = torch.Generator().manual_seed(seed)
    fv = mesh.init_state()
    x = torch.from_numpy(mesh.centers).to(dev)
    d = torch.from_numpy(np.ascontiguousarray(mesh.signdis)).to(dev).clamp(0.0, 10.0)
    layer = 1.0 - 0.8 * torch.exp(-d / 0.05)
    out = torch.from_numpy(fv).to(dev)
    for col in (0, 1, 2, 4):
        k = (torch.rand(3, 2, generator=g, dtype=torch.float64) * 4.0 - 2.0).to(dev)
        ph = (torch.rand(3, generator=g, dtype=torch.float64) * 6.28).to(dev)
        wave = sum(torch.sin(x[:, 0] * k[j, 0] + x[:, 1] * k[j, 1] + ph[j]) for j in range(3)) / 3.0
        if col in (0, 4):
            out[:, col] *= 1.0 + 0.004 * wave
        else:
            out[:, col] += 0.01 * wave
    out[:, 1] *= layer
    out[:, 2] *= layer
    a = torch.rand((), generator=g, dtype=torch.float64).item()
    nut = mesh.phys[0].nut_inf * (0.9 + 0.2 * a) * (1.0 - 0.9 * torch.exp(-d / 0.1))
    return out.cpu().numpy(), nut.cpu().numpy()


def _weights(seed):
    """Closure parameters and statistics (the layout of closure_set_params):
    a network of the trained scale whose range holds practically every cell."""
    r = np.random.default_rng(seed)
    p = np.zeros(NPARAM + 34, np.float32)
    p[:512] = r.normal(0.0, (2.0 / 8) ** 0.5, 512)
    p[512:576] = r.normal(0.0, 0.05, 64)
    p[576:4672] = r.normal(0.0, (2.0 / 64) ** 0.5, 4096)
    p[4672:4736] = r.normal(0.0, 0.05, 64)
    p[4736:4800] = r.normal(0.0, (1.0 / 64) ** 0.5, 64)
    s = p[NPARAM:]
    s[0:8], s[8:16] = FMEAN, FSTD
    s[16:24], s[24:32] = -30.0, 30.0
    s[32], s[33] = 0.02, 0.02
    return p


def prepare(case, seed):
    kind = case["kind"]
    if kind == "infer":
        mesh = _mesh("naca0012", 2, 64, 4, 1, 1)
        eng = ibgpu.Engine(mesh, mode="mixed", nstage=4, turbulence=True)
        eng.closure_init(1024)
        eng.closure_set_params(_weights(seed))
        r = np.random.default_rng(seed + 1)
        x = (np.array(FMEAN) + np.array(FSTD) * r.normal(0.0, 1.0, (case["rows"], 8))).astype(np.float32)
        return {"kind": kind, "eng": eng, "x": x}
    if kind == "train":
        mesh = _mesh("naca0015", 2, case["base"], case["levels"], 1, 1)
        eng = ibgpu.Engine(mesh, mode="fp64", nstage=4, turbulence=True)
        fv, nut = _flow(mesh, seed)
        eng.set_state(fv)
        eng.set_nut(nut)
        eng.closure_init(case["rows"], seed)
        n, k = 0, 0
        while n < case["rows"] and k < 256:      # the sampling passes of a run
            n = eng.closure_sample(0.9, 1000 + seed + k)
            k += 1
        eng.closure_fit_stats(0.0)
        return {"kind": kind, "eng": eng, "case": dict(case), "seed": seed, "start": eng.closure_params()}
    if kind == "regrid":
        meshes = [_mesh("naca0015", 2, case["base"], case["levels"], 1, 1, a) for a in (0.0, case["angle"])]
        eng = ibgpu.Engine(meshes[0], mode="mixed", nstage=4, turbulence=True)
        fv, nut = _flow(meshes[0], seed)
        eng.set_state(fv)
        eng.set_nut(nut)
        eng.upload_surface()
        return {"kind": kind, "eng": eng, "meshes": meshes, "at": 0}
    mesh = _mesh_of(case)
    eng = ibgpu.Engine(mesh, mode=case["mode"], nstage=case["stages"], temporal_refine=case["subcycle"],
                       limiter=case["limiter"], turbulence=case["closure"] != "laminar",
                       reflux=case["reflux"])
    if case["moving"]:
        eng.upload_surface()
    if case["closure"] == "learned":
        eng.closure_init(1024)
        eng.closure_set_params(_weights(seed))
        eng.closure_enable(True)
    fv, nut = _flow(mesh, seed)
    dt0 = np.array([mesh.phys[c].dt_init for c in range(mesh.ncases)])
    if not case["stepwise"]:
        if case["moving"]:
            eng.set_motion([MOTION] * mesh.ncases, t0=0.0)
        eng.prepare_march(0, case["steps"])
    return {"kind": kind, "eng": eng, "case": dict(case), "fv": fv, "nut": nut, "dt0": dt0}


# ---------------------------------------------------------------------- run
def _take(eng, case):
    """The run's results.  The mixed mode forms its fluxes and its working
    state in 32 bits, so its fields are kept as a 32-bit snapshot, as they
    are stored for post-processing."""
    fv = eng.get_state()
    linf, l2 = eng.ResinDomain()
    out = {"state": fv, "force": eng.ComptWallForce(), "dt": eng.get_dt(), "linf": linf, "l2": l2}
    if case["closure"] != "laminar":
        out["nut"] = eng.get_nut()
    if case["mode"] == "mixed":
        out = {k: torch.from_numpy(v).to(torch.float32) for k, v in out.items()}
    return out


def run(state):
    eng = state["eng"]
    if state["kind"] == "infer":
        return eng.closure_infer(state["x"])
    if state["kind"] == "train":
        c = state["case"]
        eng.closure_set_params(state["start"])
        loss = eng.closure_train(c["steps"], batch=c["batch"], lr=1e-3, seed=state["seed"])
        return {"loss": np.float32(loss), "params": eng.closure_params()}
    if state["kind"] == "regrid":
        state["at"] ^= 1
        eng.regrid(state["meshes"][state["at"]])
        return {"state": torch.from_numpy(eng.get_state()).to(torch.float32),
                "nut": torch.from_numpy(eng.get_nut()).to(torch.float32)}
    case = state["case"]
    eng.set_state(state["fv"])
    if case["closure"] != "laminar":
        eng.set_nut(state["nut"])
    eng.set_dt(state["dt0"])
    if case["moving"]:
        eng.set_motion([MOTION] * eng.mesh.ncases, t0=0.0)
    if case["stepwise"]:
        hist = []
        for ts in range(case["steps"]):
            eng.TimeMarching(ts, 1)
            hist.append(eng.ResinDomain()[0])
        out = _take(eng, case)
        hist = torch.from_numpy(np.array(hist))
        out["history"] = hist.to(torch.float32) if case["mode"] == "mixed" else hist
        return out
    eng.TimeMarching(0, case["steps"], use_graph=True)
    return _take(eng, case)


# --------------------------------------------------------------------- work
def _cell_stages(case):
    """(cell-stages, cell-steps) of a march: the normal cells of the levels
    each step marches."""
    mesh = _mesh_of(case)
    per = [sum(row[l] for row in mesh.counts()) for l in range(mesh.nlevels)]
    n = 0
    for ts in range(case["steps"]):
        n += sum(per[l] for l in range(mesh.nlevels)
                 if not case["subcycle"] or ts % (1 << (mesh.nlevels - 1 - l)) == 0)
    return n * case["stages"], n


def work(case):
    kind = case["kind"]
    if kind == "infer":
        return {"bytes": case["rows"] * 36.0, "flops": case["rows"] * 2.0 * (8 * 64 + 64 * 64 + 64)}
    if kind == "train":
        per = 2.0 * (8 * 64 + 64 * 64 + 64)
        return {"bytes": case["steps"] * (case["batch"] * 36.0 + NPARAM * 4.0 * 6),
                "flops": case["steps"] * case["batch"] * 3.0 * per}
    if kind == "regrid":
        n = _mesh("naca0015", 2, case["base"], case["levels"], 1, 1, 0.0).ncells
        # state and working variable out and in, the new level set's cells,
        # neighbours and faces in
        return {"bytes": n * (2 * 8 * 8.0 + 8 * 4 + 2 * 33 + 20), "flops": 0.0}
    stages, cells = _cell_stages(case)
    nv, s = case["dim"] + 2, 8 if case["mode"] == "fp64" else 4
    sa = case["closure"] != "laminar"
    # per cell-stage: the state read and written, the step-start state and
    # the frozen viscous residual read; with the closure its variable, its
    # start value, the face term and the wall distance
    b = stages * (2 * nv * s + nv * 8 + nv * s + ((2 * s + 8 + 2 * s) if sa else 0))
    # per step: the viscous pass reads the state and writes its residual
    b += cells * (2 * nv * s + (2 * s if sa else 0))
    f = stages * (500.0 if case["dim"] == 2 else 850.0) + cells * (250.0 if case["dim"] == 2 else 500.0)
    if case["closure"] == "learned":
        f += stages * 2.0 * (8 * 64 + 64 * 64 + 64)
    return {"bytes": float(b), "flops": float(f)}


# -------------------------------------------------------------------- exact
def exact(case, seed):
    """The network in 64 bits.  A march, a training run and a regrid's
    interpolation have no value outside a solver of their own."""
    if case["kind"] != "infer":
        return None
    p = _weights(seed).astype(np.float64)
    r = np.random.default_rng(seed + 1)
    x = (np.array(FMEAN) + np.array(FSTD) * r.normal(0.0, 1.0, (case["rows"], 8))).astype(np.float32)
    t = torch.from_numpy
    s = p[NPARAM:]
    h = (t(x.astype(np.float64)) - t(s[0:8])) / t(s[8:16])
    h = torch.relu(h @ t(p[:512].reshape(8, 64)) + t(p[512:576]))
    h = torch.relu(h @ t(p[576:4672].reshape(64, 64)) + t(p[4672:4736]))
    y = h @ t(p[4736:4800]) + float(p[4800])
    return float(s[32]) + float(s[33]) * y
