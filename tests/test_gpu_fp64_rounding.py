"""Rounding error of the FP64 face fluxes against 80-bit arithmetic.

The FP64 kernels replace quotients and roots by refined reciprocals and fuse
products with sums.  The same formulas are evaluated here in 80 bits (the
exact value) and in 64 bits with a rounding after every operation; the engine
may be no further from the exact value than the latter, and for the inviscid
flux, half of whose additions are fused, 10 % closer.
"""
import numpy as np
import pytest

import ibgpu
from test_gpu_parity import perturbed_state

pytestmark = [pytest.mark.gpu, pytest.mark.skipif(np.finfo(np.longdouble).nmant < 63, reason="no 80-bit long double")]


class Faces:
    """The stencils of a mesh's faces."""

    def __init__(self, mesh):
        self.mesh, self.d = mesh, mesh.face_dir.astype(int)
        self.lo, self.hi = mesh.face_cells[:, 0].astype(int), mesh.face_cells[:, 1].astype(int)
        e = np.eye(3, dtype=int)
        nb = lambda c, o: mesh.nb[c, (o[..., 0] + 1) * 9 + (o[..., 1] + 1) * 3 + o[..., 2] + 1]
        back, ahead = nb(self.lo, -e[self.d]), nb(self.hi, e[self.d])
        self.ll, self.rr = np.where(back < 0, ahead, back), np.where(ahead < 0, back, ahead)
        self.tan = {}     # axis -> (faces of another direction, their four cells)
        for t in range(mesh.dim):
            m = np.flatnonzero(self.d != t)
            self.tan[t] = m, [nb(c[m], s * e[t]) for s in (1, -1) for c in (self.lo, self.hi)]
        block = np.repeat(np.arange(len(mesh.blk_h)), np.diff(mesh.blk_face_start))
        self.h = mesh.blk_h[block]
        self.area = np.choose(self.d, [self.h[:, 1] * self.h[:, 2], self.h[:, 2] * self.h[:, 0], self.h[:, 0] * self.h[:, 1]])


def inviscid(F, q, P, limiter, R):
    """All-speed Roe flux (mass, momenta, energy) from (roe, u, v, w, p)."""
    gama, Rg, Cv, Ma = R(P.gama), R(P.Rg), R(P.Cv), R(P.Ma)
    n, area, half = np.arange(len(F.d)), F.area.astype(R), R(0.5)

    def slope(a, b):
        with np.errstate(all="ignore"):
            r = b / a
            r = np.where((np.abs(r) > 1e10) | np.isnan(r), np.where(b > 0, R(1e6), R(-1)), r)
        r = np.maximum(r, R(0))
        return half * a * ((r * r + r) / (r * r + 1) if limiter else 2 * r / (1 + r))

    jump = q[F.hi] - q[F.lo]
    l = q[F.lo] + slope(q[F.lo] - q[F.ll], jump)
    r = q[F.hi] - slope(q[F.rr] - q[F.hi], jump)
    normal = np.zeros((len(n), 3), R)
    normal[n, F.d] = 1
    side = []
    for s in (l, r):
        T, v = s[:, 4] / (s[:, 0] * Rg), s[n, 1 + F.d]
        e = Cv * T + half * (s[:, 1] * s[:, 1] + s[:, 2] * s[:, 2] + s[:, 3] * s[:, 3])
        mom = s[:, :1] * s[:, 1:4] * v[:, None] + s[:, 4:] * normal
        side.append((T, v, e, np.column_stack([s[:, 0] * v, mom, (s[:, 4] + e * s[:, 0]) * v])))
    (lT, lv, le, lf), (rT, rv, re, rf) = side
    root = np.sqrt(r[:, 0] / l[:, 0])
    w, a_roe = 1 / (1 + root), np.sqrt(l[:, 0] * r[:, 0])
    vel = (l[:, 1:4] + r[:, 1:4] * root[:, None]) * w[:, None]
    h = ((le + l[:, 4] / l[:, 0]) + (re + r[:, 4] / r[:, 0]) * root) * w
    c = np.sqrt((gama - 1) * (h - (vel[:, 0] * vel[:, 0] + vel[:, 1] * vel[:, 1] + vel[:, 2] * vel[:, 2]) / 2))
    c2, un = c * c, vel[n, F.d]
    dr, dp, du, dn = r[:, 0] - l[:, 0], r[:, 4] - l[:, 4], r[:, 1:4] - l[:, 1:4], rv - lv
    f = np.abs((lv + rv) * half / np.sqrt(gama * Rg * ((lT + rT) * half)))
    f = np.minimum(np.maximum(f, Ma), R(1))
    n0 = np.sqrt(4 * c * c * f + (1 - f) * (1 - f) * un * un)
    n1, n2 = np.abs(half * ((1 + f) * un + n0)), np.abs(half * ((1 + f) * un - n0))
    k, fa = 1 / (2 * c2) * area, area * np.abs(un)
    al0 = fa * (dr - dp / c2)
    al1, al2 = k * n1 * (dp + a_roe * c * dn), k * n2 * (dp - a_roe * c * dn)
    al3, al4 = al0 + al1 + al2, c * (al1 - al2)
    al5 = fa[:, None] * (a_roe[:, None] * (du - normal * dn[:, None]))
    en = h * al3 + un * al4 + (vel * al5).sum(1) - c2 / (gama - 1) * al0
    up = np.column_stack([al3, vel * al3[:, None] + normal * al4[:, None] + al5, en])
    return (lf + rf) * (half * area)[:, None] - up


def viscous(F, q, P, R):
    """Laminar viscous flux (momenta, energy)."""
    n, area = np.arange(len(F.d)), F.area.astype(R)
    T = q[:, 4] / (q[:, 0] * R(P.Rg))
    V = np.column_stack([q[:, 1:4], T])
    G = np.zeros((len(n), 4, 3), R)
    for t, (m, (a, b, c, d)) in F.tan.items():
        G[m, :, t] = (V[a] + V[b] - V[c] - V[d]) * R(0.25)
    G[n, :, F.d] = V[F.hi] - V[F.lo]
    G *= (1 / F.h).astype(R)[:, None, :]
    S, ft = R(P.S_over_T_ref), (T[F.lo] + T[F.hi]) * R(0.5)
    mu = np.sqrt(ft * ft * ft) * ((1 + S) / (ft + S))
    div = G[:, 0, 0] + G[:, 1, 1] + G[:, 2, 2]
    tau = np.empty((len(n), 3), R)
    for j in range(3):
        shear = mu / R(P.Re) * (G[n, j, F.d] + G[n, F.d, j])
        tau[:, j] = np.where(F.d == j, 2 * mu * (G[:, j, j] - div / 3) / R(P.Re), shear)
    vel = (q[F.lo, 1:4] + q[F.hi, 1:4]) * R(0.5)
    work = (vel * tau).sum(1) + R(P.qk) * mu * G[n, 3, F.d]
    return np.column_stack([tau, work]) * area[:, None]


@pytest.mark.parametrize("dim,limiter", [(2, 0), (2, 1), (3, 0), (3, 1)])
def test_flux_error_against_80_bits(dim, limiter):
    mesh = ibgpu.Mesh(ibgpu.tiny_case(Re=2000.0) if dim == 2 else ibgpu.tiny3d_case())
    P, F, R80 = mesh.phys[0], Faces(mesh), np.longdouble
    eng = ibgpu.Engine(mesh, mode="fp64", limiter=limiter)
    cols = [0, 1, 2, 4] if dim == 2 else [0, 1, 2, 3, 4]
    vcols = [k - 1 for k in cols[1:]]
    err = []
    for seed in range(4):
        fv, r = perturbed_state(mesh, seed=seed), np.random.default_rng(seed)
        fv[:, [0, 4]] *= 1.0 + 0.05 * r.uniform(-1, 1, (mesh.ncells, 2))
        fv[:, 1:1 + dim] += 0.05 * r.uniform(-1, 1, (mesh.ncells, dim))
        eng.set_state(fv)
        q, q80 = fv[:, :5], fv[:, :5].astype(R80)
        exact = inviscid(F, q80, P, limiter, R80), viscous(F, q80, P, R80)
        plain = inviscid(F, q, P, limiter, np.float64), viscous(F, q, P, np.float64)
        got = eng.faceflux(), eng.vsflux()[:, 1:]
        size = [np.sqrt((e.astype(float) ** 2).mean(0)) for e in exact]
        mean = lambda a: [(((x - e).astype(float)[:, k] / s[k]) ** 2).mean(0)
                          for x, e, s, k in zip(a, exact, size, (cols, vcols))]
        err.append(mean(got) + mean(plain))
    gi, gv, pi, pv = (np.sqrt(np.mean(e, 0)) for e in zip(*err))
    print("inviscid", gi, "plain", pi, "viscous", gv, "plain", pv)
    # (2 %: the scatter of a mean over some 1e4 faces and four states)
    assert (gi <= 0.9 * 1.02 * pi).all()
    assert (gv <= 1.02 * pv).all()
