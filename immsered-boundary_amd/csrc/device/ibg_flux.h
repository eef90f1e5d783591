// ibg_flux.h — per-face arithmetic of the residual engine (device side).
//
// Templated on the arithmetic type R (double: plain mode; float: mixed mode)
// and on the dimension D (2: the w component is identically zero and all of
// its terms are dropped, which is exact because every one of them is a
// product with w = 0 or a zero metric component).
#pragma once
#include <hip/hip_runtime.h>

#include <type_traits>

#include "ibg_common.h"

namespace ibg {

__device__ __forceinline__ double r_abs(double x) { return fabs(x); }
__device__ __forceinline__ float r_abs(float x) { return fabsf(x); }

// Reciprocal, quotient and square root of the flux arithmetic.  FP32: the
// hardware v_rcp_f32 / v_sqrt_f32 (~1 ulp).  FP64: the hardware estimate
// refined.  A zero, denormal or infinite divisor (or root) gives NaN: the
// places that meet one in earnest keep it in range or divide with '/' (the
// limiters' sums of tiny differences, the eigenvalues' root at rest, S~ of a
// uniform stream, a wall infinitely far away, an infinite Reynolds number).
__device__ __forceinline__ float f_rcp(float x) { return __builtin_amdgcn_rcpf(x); }
__device__ __forceinline__ float f_sqrt(float x) { return __builtin_amdgcn_sqrtf(x); }
__device__ __forceinline__ float n_div(float n, float x) { return n * f_rcp(x); }
// FP64 quotient: two Newton steps and Markstein's fused residual, the IEEE
// sequence without its range scaling and fixup: the same value in the normal
// range.
__device__ __forceinline__ double n_div(double n, double x) {
#pragma clang fp contract(off)
  double y = __builtin_amdgcn_rcp(x);
  y = fma(fma(-x, y, 1.0), y, y);
  y = fma(fma(-x, y, 1.0), y, y);
  const double q = n * y;
  return fma(fma(-x, q, n), y, q);
}
// The same by a constant c of reciprocal ic.
__device__ __forceinline__ double c_div(double n, double c, double ic) {
#pragma clang fp contract(off)
  const double q = n * ic;
  return fma(fma(-c, q, n), ic, q);
}
// FP64 reciprocal and roots to half a unit in the last place (and 2^-18 of
// one): v_rcp_f64 and v_rsq_f64 are good to 2^-24 (measured on gfx950:
// 2^-24.4 and 2^-24.2), so one step of third order (e + e^2, e/2 + 3/8 e^2) on
// an exact error e reaches 2^-72, and so does a step of second order followed
// by one with the exact residual x - g^2.
__device__ __forceinline__ double n_rcp(double x) {
#pragma clang fp contract(off)
  const double y = __builtin_amdgcn_rcp(x);
  const double e = fma(-x, y, 1.0);
  return fma(y, fma(e, e, e), y);
}
__device__ __forceinline__ double n_sqrt(double x) {   // x > 0
#pragma clang fp contract(off)
  const double y = __builtin_amdgcn_rsq(x), h = 0.5 * y;
  double g = x * y;
  g = fma(g, fma(-h, g, 0.5), g);
  return fma(fma(-g, g, x), h, g);
}
// the same of a value that may be zero (not of a negative one)
__device__ __forceinline__ double n_sqrt0(double x) {
#pragma clang fp contract(off)
  const double y = __builtin_amdgcn_rsq(fmax(x, 0x1p-1000)), h = 0.5 * y;
  double g = x * y;
  g = fma(g, fma(-h, g, 0.5), g);
  return fma(fma(-g, g, x), h, g);
}
__device__ __forceinline__ double n_rsqrt(double x) {   // x > 0
#pragma clang fp contract(off)
  const double y = __builtin_amdgcn_rsq(x), t = x * y, tl = fma(x, y, -t);
  const double e = fma(-tl, y, fma(-t, y, 1.0));
  return fma(y * e, fma(e, 0.375, 0.5), y);
}

// Physical constants of one case in the arithmetic type of the kernel.
template <typename R>
struct PhysR {
  R gama, Rg, Cv, Ma;
  R gm1, ig1;    // gama - 1 and its reciprocal
  R iRg;         // 1 / Rg (FP32 only)
  R cpR;         // Cv / Rg + 1: enthalpy h = cpR p / roe + |u|^2 / 2
  R cpRl;        // what its rounding left out (FP64 only)
};
template <typename R, class Q>
__device__ __forceinline__ PhysR<R> phys_r(const Q &P) {
  PhysR<R> ph;
  ph.gama = (R)P.gama; ph.Rg = (R)P.Rg; ph.Cv = (R)P.Cv; ph.Ma = (R)P.Ma;
  ph.cpR = (R)P.cpR;
  if constexpr (sizeof(R) == 4) {
    ph.gm1 = ph.gama - 1.0f; ph.ig1 = f_rcp(ph.gm1); ph.iRg = f_rcp(ph.Rg); ph.cpRl = 0.0f;
  } else {
    ph.gm1 = P.gama - 1.0; ph.ig1 = P.ig1; ph.iRg = 0.0; ph.cpRl = P.cpRl;
  }
  return ph;
}
// the same from the table of the FP32 constants
template <class Q>
__device__ __forceinline__ PhysR<float> phys_r32(const Q &F) {
  return PhysR<float>{F.gama, F.Rg, F.Cv, F.Ma, F.gm1, F.ig1, F.iRg, F.cpR, 0.0f};
}

template <typename R, int D>
struct Prim {
  R r, u, v, w, p;   // w unused when D == 2
};

// Limited half slope 0.5 a phi(r), r = b / a, of SlopeCorrection_Left/Right
// (Slopelimiter.H:22-58, comptqleft/right NS_Solver.H:21-27): left of a face
// a = qi - q_i, b = qi1 - qi, added to qi; right of it a = qi1 - qi,
// b = qi - q_i, subtracted.  With one division, as a product of a weight and
// b or a + b: for a and b of one sign (r > 0)
//   van Leer   phi = 2r/(1+r):        0.5 a phi = |a| / (|a| + |b|)  b
//   van Albada phi = (r^2+r)/(r^2+1): 0.5 a phi = 0.5 |a| |b| / (a^2 + b^2)  (a + b)
// and 0 otherwise (the reference forms r and phi with a division each): the
// weight has max(a sign(b), 0) for |a|.
// No intermediate leaves the range of a normal number, whatever the size of
// a and b: the front of a disturbance in a uniform stream decays from cell to
// cell through differences of 1e-100, 1e-200 and less, whose products and
// square sums are denormal or zero and whose reciprocal is infinite.  So the
// signs are compared as such, van Leer's divisor has an addend of 2^-1021
// (lost in rounding above 2^-967), and van Albada's squares are formed of
// |a| and |b| scaled to at most one by a power of two.
// A NaN or infinite difference gives NaN.  Van Leer's weight takes no more
// instructions than the form a b / (a + b), whose product cannot fuse with the
// cell value (the moving 2D section, 128 steps, 70.8 -> 70.0 ms), van Albada's
// four more a slope (the mid-size laminar case 5.30 -> 5.33 ms).
// The reference's guard, |r| > 1e10 or NaN: r becomes 1e6 for b > 0, else
// -1, so phi is 1e6's or 0 whatever the sign of a.
// fixed_slope is the value where the guard holds.  That needs a jump beside
// a difference 1e10 times smaller, flow uniform but for rounding: the waves
// that meet one take a second pass over the limiters (muscl_guarded).
struct HalfSlope {
  double w, d;   // the half slope as a product
};
// a sign(b)
__device__ __forceinline__ double along(double a, double b) {
  return __hiloint2double(__double2hiint(a) ^ (__double2hiint(b) & (int)0x80000000), __double2loint(a));
}
// s = a sign(b) in the place of a
template <bool ALBADA>
__device__ __forceinline__ HalfSlope half_slope(double s, double b) {
#pragma clang fp contract(off)
  double m;
  asm("v_max_f64 %0, %1, 0" : "=v"(m) : "v"(s));   // (fmax would quiet s first; 0 for a NaN)
  const double y = r_abs(b);
  if (ALBADA) {
    const int k = -__builtin_amdgcn_frexp_exp(r_abs(s) + y);
    const double u = __builtin_ldexp(m, k), v = __builtin_ldexp(y, k);
    return {0.5 * u * v * n_rcp(fma(u, u, fma(v, v, 0x1p-1000))), along(s, b) + b};
  }
  return {m * n_rcp(r_abs(s) + (y + 0x1p-1021)), b};
}
template <bool ALBADA>
__device__ __forceinline__ double fixed_slope(double a, double b) {
#pragma clang fp contract(off)
  const double phi = ALBADA ? (1.0e12 + 1.0e6) / (1.0e12 + 1.0) : 2.0e6 / (1.0 + 1.0e6);
  return (b > 0.0) ? 0.5 * a * phi : 0.0;
}
__device__ __forceinline__ bool slope_guard(double a, double b) { return r_abs(b) > 1.0e10 * r_abs(a); }
// Left and right values of one variable; guard: whether the reference's
// guard holds on either side.
template <bool ALBADA>
__device__ __forceinline__ void muscl(double q0, double q1, double q2, double q3, double &left,
                                      double &right, bool &guard) {
#pragma clang fp contract(off)
  const double d0 = q1 - q0, d1 = q2 - q1, d2 = q3 - q2;
  const double s0 = along(d0, d1), s2 = along(d2, d1);
  const HalfSlope l = half_slope<ALBADA>(s0, d1), r = half_slope<ALBADA>(s2, d1);
  left = fma(l.w, l.d, q1);
  right = fma(-r.w, r.d, q2);
  guard = guard | slope_guard(s0, d1) | slope_guard(s2, d1);
}
template <bool ALBADA>
__device__ __forceinline__ void muscl_guarded(double q0, double q1, double q2, double q3,
                                              double &left, double &right) {
#pragma clang fp contract(off)
  const double d0 = q1 - q0, d1 = q2 - q1, d2 = q3 - q2;
  if (slope_guard(along(d0, d1), d1)) left = q1 + fixed_slope<ALBADA>(d0, d1);
  if (slope_guard(along(d2, d1), d1)) right = q2 - fixed_slope<ALBADA>(d2, d1);
}

// All-speed Roe flux of one face from the 4-cell stencil (t0,t1 | t2,t3),
// the body of ComputeFaceFlux NS_Solver.H:766-794 with FaceLeftRight
// (:31-45), Get_inv_flux (FlowVariables.H:59-64), Roeaverage (:51-62),
// roe0c_coef ROE_ALLSPEED (:66-77) and ComptFaceFlux (:87-113), the upwind
// term without the factor 1/2 as in the reference.  In the face's own frame:
// u is the normal velocity, v (and w) the tangential ones, so the normal's
// products with 0 and 1 are gone, and the terms of the tangential jump
// along the normal (du_n - dubar = 0) with them.  Energy and temperature
// enter as p/roe only: gama Rg T = gama p/roe, and roe e + p = cpR p +
// roe |u|^2/2 needs no quotient.  Per face 4 reciprocals, 4 roots and the 2 NV
// limiter quotients; the reference's form has 26 divisions and 5 roots (2D),
// in FP64 each a chain of 10 to 15 instructions, and the kernels were bound
// by their FP64 issue.  With the SA functions below: 128 steps of the moving
// 2.6M-cell 2D section 127.7 -> 99.4 ms, 32 steps of the 2.7M-cell 3D section
// 70.2 -> 57.0 ms; with third-order reciprocals and the guard out of the common
// path the stage launches go from 134 to 118 us (2D) and from 294 to 242 us
// (3D, both with block tiles).
// rms error against 80-bit arithmetic over the faces of small 2D (3D) sections
// with jumps of a percent between cells, relative to the rms flux, the
// 26-division form -> this one: mass 1.08e-16 -> 1.08e-16 (1.60 -> 1.60),
// normal momentum 0.82 -> 0.81 (0.95 -> 0.95), energy 1.28 -> 1.21 (1.67 ->
// 1.61).  The energy is the component that is easily lost: formed from p/roe,
// with the rounded constant Cv/Rg + 1, it had 1.43 (1.80).
// The fused operations are written out here and in the viscous flux below, so
// that block and general tiles, whose faces have a known direction or not,
// round alike and the tile size does not change a bit of the results.
// Output: (mass, normal, tangential momenta, energy).
template <int D>
__device__ __forceinline__ void roe_normal(const Prim<double, D> &t0, const Prim<double, D> &t1,
                                           const Prim<double, D> &t2, const Prim<double, D> &t3, double area,
                                           const PhysR<double> &ph, int lim, double *flux) {
#pragma clang fp contract(off)
  double lr, rr, lu, ru, lv, rv, lw = 0.0, rw = 0.0, lp, rp;
  auto reconstruct = [&](auto albada) {
    constexpr bool A = decltype(albada)::value;
    bool guard = false;
    muscl<A>(t0.r, t1.r, t2.r, t3.r, lr, rr, guard);
    muscl<A>(t0.u, t1.u, t2.u, t3.u, lu, ru, guard);
    muscl<A>(t0.v, t1.v, t2.v, t3.v, lv, rv, guard);
    if (D == 3) muscl<A>(t0.w, t1.w, t2.w, t3.w, lw, rw, guard);
    muscl<A>(t0.p, t1.p, t2.p, t3.p, lp, rp, guard);
    if (__any(guard)) {
      muscl_guarded<A>(t0.r, t1.r, t2.r, t3.r, lr, rr);
      muscl_guarded<A>(t0.u, t1.u, t2.u, t3.u, lu, ru);
      muscl_guarded<A>(t0.v, t1.v, t2.v, t3.v, lv, rv);
      if (D == 3) muscl_guarded<A>(t0.w, t1.w, t2.w, t3.w, lw, rw);
      muscl_guarded<A>(t0.p, t1.p, t2.p, t3.p, lp, rp);
    }
  };
  if (lim == 1) reconstruct(std::true_type());   // lim is uniform: one branch a face
  else reconstruct(std::false_type());
  const double ilr = n_rcp(lr);
  double lq = fma(lu, lu, lv * lv), rq = fma(ru, ru, rv * rv);
  if (D == 3) { lq = fma(lw, lw, lq); rq = fma(rw, rw, rq); }
  // roe h per volume, formed without the quotient p / roe
  const double el = fma(ph.cpR, lp, fma(ph.cpRl, lp, (0.5 * lr) * lq));
  const double er = fma(ph.cpR, rp, fma(ph.cpRl, rp, (0.5 * rr) * rq));
  const double irr = n_rcp(rr);
  const double hl = el * ilr, hr = er * irr;
  // central part 1/2 (F_L + F_R) A, without the factor A/2
  const double ml = lr * lu, mr = rr * ru;
  const double ha = 0.5 * area;
  const double c0 = fma(lr, lu, mr);
  const double c1 = fma(ml, lu, lp) + fma(mr, ru, rp);
  const double c2 = fma(ml, lv, mr * rv);
  const double c4 = fma(el, lu, er * ru);
  const double droe = rr - lr, dp = rp - lp, dubar = ru - lu;
  // Roe average: sqrt(rr / lr) = sqrt(lr rr) / lr
  const double a_roe = n_sqrt(lr * rr);
  const double q = a_roe * ilr;
  const double wl = n_rcp(1.0 + q);
  const double a_u = fma(ru, q, lu) * wl;
  const double a_v = fma(rv, q, lv) * wl;
  const double a_w = (D == 3) ? fma(rw, q, lw) * wl : 0.0;
  const double a_h = fma(hr, q, hl) * wl;
  double q2 = fma(a_u, a_u, a_v * a_v);
  if (D == 3) q2 = fma(a_w, a_w, q2);
  const double csq = ph.gm1 * fma(-0.5, q2, a_h);
  const double a_c = n_sqrt(csq);
  const double icsq = n_rcp(csq);
  const double faa = area * r_abs(a_u);
  const double coef12 = (0.5 * ha) * icsq;   // times 2 n1, 2 n2
  const double rc = a_roe * a_c;
  const double al0 = faa * fma(-dp, icsq, droe);
  // all-speed eigenvalues (NS_Solver.H:66-77): f = min(max(Ma_face, Ma_inf), 1)
  double f = r_abs((lu + ru) * 0.5) * n_rsqrt(ph.gama * (fma(rp, irr, lp * ilr) * 0.5));
  f = f < ph.Ma ? ph.Ma : f;
  f = f > 1.0 ? 1.0 : f;
  const double g = (1.0 - f) * a_u, f1 = 1.0 + f;
  const double n0 = n_sqrt0(fma(4.0 * csq, f, g * g));   // 0 at rest where Ma_inf is 0
  const double n1 = coef12 * r_abs(fma(f1, a_u, n0));
  const double n2 = coef12 * r_abs(fma(f1, a_u, -n0));
  const double x1 = fma(rc, dubar, dp), x2 = fma(-rc, dubar, dp);
  const double al3 = fma(n2, x2, fma(n1, x1, al0));
  const double al4 = a_c * fma(n1, x1, -(n2 * x2));
  const double fr = faa * a_roe;
  const double al6 = fr * (rv - lv);
  const double al7 = (D == 3) ? fr * (rw - lw) : 0.0;
  flux[0] = fma(c0, ha, -al3);
  flux[1] = fma(c1, ha, -fma(a_u, al3, al4));
  flux[2] = fma(c2, ha, -fma(a_v, al3, al6));
  double en = fma(a_h, al3, a_u * al4);
  en = fma(a_v, al6, en);
  if (D == 3) en = fma(a_w, al7, en);
  en = fma(-(csq * ph.ig1), al0, en);
  if (D == 3) flux[3] = fma(fma(ml, lw, mr * rw), ha, -fma(a_w, al3, al7));
  flux[D == 3 ? 4 : 3] = fma(c4, ha, -en);
}

// Into and out of the frame of a face of direction dir: the normal velocity
// (momentum) changes places with u.
template <int D>
__device__ __forceinline__ Prim<double, D> to_face(const Prim<double, D> &q, int dir) {
  Prim<double, D> o = q;
  o.u = dir == 0 ? q.u : ((D == 3 && dir == 2) ? q.w : q.v);
  o.v = dir == 1 ? q.u : q.v;
  if (D == 3) o.w = dir == 2 ? q.u : q.w;
  return o;
}
template <int D>
__device__ __forceinline__ void from_face(double *f, int dir) {
  const double n = f[1], t = f[2];
  f[1] = dir == 0 ? n : ((D == 3 && dir == 2) ? f[3] : t);
  f[2] = dir == 1 ? n : t;
  if (D == 3) f[3] = dir == 2 ? n : f[3];
}

// Flux of an axis-aligned face.  Output: D == 2: (mass, x-mom, y-mom,
// energy); D == 3: (mass, x, y, z momentum, energy).  DIR, FLAT: as the FP32
// form below, which the tiles call alike (FLAT changes nothing here).
template <int D, int DIR = -1, bool FLAT = false>
__device__ __forceinline__ void roe_flux(const Prim<double, D> &t0, const Prim<double, D> &t1,
                                         const Prim<double, D> &t2, const Prim<double, D> &t3,
                                         int dir, double area, const PhysR<double> &ph, int lim,
                                         double *flux) {
  if (DIR >= 0) dir = DIR;
  roe_normal<D>(to_face<D>(t0, dir), to_face<D>(t1, dir), to_face<D>(t2, dir), to_face<D>(t3, dir),
                area, ph, lim, flux);
  from_face<D>(flux, dir);
}

// ---------------------------------------------------------------------------
// Mixed-mode (FP32) form of the same face flux.  The arithmetic is the same
// expression set, evaluated with the hardware reciprocal and square root
// (v_rcp_f32, v_sqrt_f32, ~1 ulp) and with the van Leer limiter in its
// one-reciprocal form: for r = dqii/dqi > 0,
//   qi + 0.5 dqi phi(r) = qi + dqi dqii / (dqi + dqii),
// and qi otherwise (the reference's 1e10/1e6 guards only matter when
// |dqi| < 1e-10 |dqii|, where both forms give qi to within 1e-10 dqii).
// The error of this mode against the FP64 oracle is measured, not assumed.

// Limited half slope 0.5 a phi(b / a) of FP32 (see half_slope above), as the
// value q + or - it.  van Albada through the ratio r (as the reference forms
// it, with its guards): r > 0 here, phi = (r^2 + r)/(r^2 + 1).  The
// one-reciprocal form pr (a + b) / (a^2 + b^2) overflows in FP32 once both
// differences fall below ~1e-19 (the square sum below 2^-126).
__device__ __forceinline__ float fast_albada(float num, float den) {
  float r = num * f_rcp(den);
  if (!(r <= 1.0e10f)) r = (num > 0.0f) ? 1000000.0f : 0.0f;   // also NaN / inf
  return fmaf(r, r, r) * f_rcp(fmaf(r, r, 1.0f));
}
// The same without branches, for the block tiles: a wave's lanes mostly have
// both signs, so the branches only cost (stage 60.6 -> 56.4 us on the
// 2.6M-cell section; 3D 117 -> 111.5, once its residual sums leave the
// registers for it).  In general tiles the extra live values cost the learned
// closure its occupancy.
template <bool kLeft, bool ALBADA>
__device__ __forceinline__ float flat_slope(float q, float a, float b) {
#pragma clang fp contract(off)
  const float pr = a * b;
  const float x = ALBADA ? fmaf(kLeft ? 0.5f * a : -0.5f * a, fast_albada(b, a), q)
                         : fmaf(kLeft ? pr : -pr, f_rcp(a + b), q);
  return pr > 0.0f ? x : q;
}
template <bool kLeft>
__device__ __forceinline__ float fast_slope(float q, float a, float b, int lim) {
#pragma clang fp contract(off)
  const float pr = a * b;
  if (!(pr > 0.0f)) return q;
  if (lim == 1) return fmaf(kLeft ? 0.5f * a : -0.5f * a, fast_albada(b, a), q);
  return fmaf(kLeft ? pr : -pr, f_rcp(a + b), q);
}

// DIR: the face's direction where the compiler knows it (block tiles), -1
// where it is dir.  The fused operations are written out, so that both forms
// round alike: the terms that a known direction drops are exact zeros and
// products with one.
// FLAT: the limiter without branches.
template <int D, int DIR = -1, bool FLAT = false>
__device__ __forceinline__ void roe_flux(const Prim<float, D> &t0, const Prim<float, D> &t1,
                                         const Prim<float, D> &t2, const Prim<float, D> &t3,
                                         int dir, float area, const PhysR<float> &ph, int lim,
                                         float *flux) {
#pragma clang fp contract(off)
  const float gama = ph.gama, Rg = ph.Rg, Cv = ph.Cv;
  float lr, rr, lu, ru, lvv, rvv, lw = 0.0f, rw = 0.0f, lp, rp;
  auto reconstruct = [&](auto m) {
    m(t0.r, t1.r, t2.r, t3.r, lr, rr);
    m(t0.u, t1.u, t2.u, t3.u, lu, ru);
    m(t0.v, t1.v, t2.v, t3.v, lvv, rvv);
    if (D == 3) m(t0.w, t1.w, t2.w, t3.w, lw, rw);
    m(t0.p, t1.p, t2.p, t3.p, lp, rp);
  };
  auto flat = [&](auto albada) {
    constexpr bool A = decltype(albada)::value;
    reconstruct([&](float q0, float q1, float q2, float q3, float &l, float &r) {
      const float d0 = q1 - q0, d1 = q2 - q1, d2 = q3 - q2;
      l = flat_slope<true, A>(q1, d0, d1);
      r = flat_slope<false, A>(q2, d2, d1);
    });
  };
  if constexpr (FLAT) {
    if (lim == 1) flat(std::true_type());   // lim is uniform: one branch a face
    else flat(std::false_type());
  } else {
    reconstruct([&](float q0, float q1, float q2, float q3, float &l, float &r) {
      const float d0 = q1 - q0, d1 = q2 - q1, d2 = q3 - q2;
      l = fast_slope<true>(q1, d0, d1, lim);
      r = fast_slope<false>(q2, d2, d1, lim);
    });
  }
  const float ilr = f_rcp(lr), irr = f_rcp(rr);
  const float iRg = ph.iRg;
  const float plr = lp * ilr, prr = rp * irr;
  const float rT = prr * iRg;
  float lq = fmaf(lu, lu, lvv * lvv), rq = fmaf(ru, ru, rvv * rvv);
  if (D == 3) { lq = fmaf(lw, lw, lq); rq = fmaf(rw, rw, rq); }
  const float le = fmaf(0.5f, lq, Cv * (plr * iRg)), re = fmaf(0.5f, rq, Cv * rT);
  auto pick = [&](float x, float y, float z) {
    if (DIR >= 0) return DIR == 0 ? x : (DIR == 1 ? y : z);
    return dir == 0 ? x : (dir == 1 ? y : z);
  };
  const float lv = pick(lu, lvv, lw), rv = pick(ru, rvv, rw);
  const float k0 = dir == 0 ? 1.0f : 0.0f, k1 = dir == 1 ? 1.0f : 0.0f, k2 = dir == 2 ? 1.0f : 0.0f;
  // k x + y with the direction's k = 0 or 1
  auto kfma = [&](int d, float k, float x, float y) {
    if (DIR >= 0) return DIR == d ? x + y : y;
    return fmaf(k, x, y);
  };
  // central part 1/2 (F_L + F_R) A
  const float ha = 0.5f * area;
  const float p0 = fmaf(lr, lv, rr * rv);
  auto mom = [&](int d, float k, float l, float r) {
    float x;
    if (DIR >= 0) x = DIR == d ? fmaf(lr * l, lv, lp) : (lr * l) * lv;
    else x = fmaf(lr * l, lv, lp * k);
    return kfma(d, k, rp, fmaf(rr * r, rv, x));
  };
  const float p1 = mom(0, k0, lu, ru), p2 = mom(1, k1, lvv, rvv);
  const float p4 = fmaf(fmaf(le, lr, lp), lv, fmaf(re, rr, rp) * rv);
  const float droe = rr - lr, dp = rp - lp;
  const float dubar = rv - lv;
  // Roe average
  const float r2lroe = f_sqrt(rr * ilr);
  const float r2l0 = f_rcp(1.0f + r2lroe);
  const float h_left = fmaf(lp, ilr, le), h_right = fmaf(rp, irr, re);
  const float a_roe = f_sqrt(lr * rr);
  const float a_u = fmaf(ru, r2lroe, lu) * r2l0;
  const float a_v = fmaf(rvv, r2lroe, lvv) * r2l0;
  const float a_w = (D == 3) ? fmaf(rw, r2lroe, lw) * r2l0 : 0.0f;
  const float a_h = fmaf(h_right, r2lroe, h_left) * r2l0;
  float q2 = fmaf(a_u, a_u, a_v * a_v);
  if (D == 3) q2 = fmaf(a_w, a_w, q2);
  const float csquare = ph.gm1 * fmaf(-0.5f, q2, a_h);
  const float a_c = f_sqrt(csquare);
  const float a_ubar = pick(a_u, a_v, a_w);
  const float icsq = f_rcp(csquare);
  const float coef12 = 0.5f * icsq * area;
  const float rc = a_roe * a_c;
  const float faa = area * fabsf(a_ubar);
  const float al0 = faa * fmaf(-dp, icsq, droe);
  // all-speed eigenvalues (NS_Solver.H:66-77)
  const float T_a = fmaf(plr, iRg, rT) * 0.5f;
  const float V_a = (lv + rv) * 0.5f;
  float f_Ma = fabsf(V_a) * f_rcp(f_sqrt(gama * Rg * T_a));
  f_Ma = f_Ma < ph.Ma ? ph.Ma : f_Ma;
  f_Ma = f_Ma > 1.0f ? 1.0f : f_Ma;
  const float s0 = (1.0f - f_Ma) * (1.0f - f_Ma);
  const float namda0 = f_sqrt(fmaf(4.0f * csquare, f_Ma, s0 * a_ubar * a_ubar));
  const float n1 = coef12 * fabsf(0.5f * fmaf(1.0f + f_Ma, a_ubar, namda0));
  const float n2 = coef12 * fabsf(0.5f * fmaf(1.0f + f_Ma, a_ubar, -namda0));
  const float x1 = fmaf(rc, dubar, dp), x2 = fmaf(-rc, dubar, dp);
  const float al3 = fmaf(n2, x2, fmaf(n1, x1, al0));
  const float al4 = a_c * fmaf(n1, x1, -(n2 * x2));
  // tangential jumps: zero along the normal
  auto jump = [&](int d, float k, float du) {
    if (DIR >= 0) return DIR == d ? 0.0f : a_roe * du;
    return a_roe * fmaf(-k, dubar, du);
  };
  const float j0 = jump(0, k0, ru - lu), j1 = jump(1, k1, rvv - lvv);
  const float j2 = (D == 3) ? jump(2, k2, rw - lw) : 0.0f;
  auto upw = [&](int d, float k, float vel, float j) {
    float t;
    if (DIR >= 0) t = DIR == d ? fmaf(vel, al3, al4) : vel * al3;
    else t = fmaf(vel, al3, k * al4);
    return (DIR >= 0 && DIR == d) ? t : fmaf(faa, j, t);
  };
  const float ig1 = ph.ig1;
  flux[0] = fmaf(p0, ha, -al3);
  flux[1] = fmaf(p1, ha, -upw(0, k0, a_u, j0));
  flux[2] = fmaf(p2, ha, -upw(1, k1, a_v, j1));
  float en = fmaf(a_h, al3, a_ubar * al4);
  if (DIR != 0) en = fmaf(a_u, faa * j0, en);
  if (DIR != 1) en = fmaf(a_v, faa * j1, en);
  if (D == 3 && DIR != 2) en = fmaf(a_w, faa * j2, en);
  en = fmaf(-(csquare * ig1), al0, en);
  if (D == 3) {
    flux[3] = fmaf(mom(2, k2, lw, rw), ha, -upw(2, k2, a_w, j2));
    flux[4] = fmaf(p4, ha, -en);
  } else {
    flux[3] = fmaf(p4, ha, -en);
  }
}

template <typename R, int D>
struct ViscPhys {
  R Rg, iRe, qk, SoT;
  R ih0, ih1, ih2;   // 1/dh
  R ar0, ar1, ar2;   // face areas
  R iqkt;            // 1 / (Re*Pr_tur*(gama-1)*Ma^2) (SA closure)
  R Re, qkt;         // (FP64 only)
};
// reciprocal of a constant divisor of the FP32 viscous terms: the hardware's,
// as every quotient of that mode
__device__ __forceinline__ float c_rcp(float x) { return f_rcp(x); }

// Spalart-Allmaras constants, Turbulence.cpp:3-19
struct SA {
  static constexpr double cb1 = 0.1355;
  static constexpr double segma = 2.0 / 3.0;
  static constexpr double cb2 = 0.622;
  static constexpr double kappa = 0.41;
  static constexpr double cw2 = 0.3;
  static constexpr double cw3 = 2.0;
  static constexpr double cv1 = 7.1;
  static constexpr double ct3 = 1.2;
  static constexpr double ct4 = 0.5;
  static constexpr double cw1 = cb1 / (kappa * kappa) + (1.0 + cb2) / segma;
  static constexpr double cv1three = cv1 * cv1 * cv1;
};

// quotient of the viscous and SA terms (divisors are positive and normal),
// and the root of a value that may be zero
template <typename R> __device__ __forceinline__ R v_div(R a, R b) { return n_div(a, b); }
template <typename R> __device__ __forceinline__ R v_sqrt(R a);
template <> __device__ __forceinline__ float v_sqrt<float>(float a) { return f_sqrt(a); }
template <> __device__ __forceinline__ double v_sqrt<double>(double a) {
  const double g = n_sqrt(a);
  return a == 0.0 ? a : g;
}
// The constants of the SA source: S/T_ref of Sutherland's law and 1 + it, the
// Reynolds number, its reciprocal (FP32) and sqrt(2).
template <typename R>
struct SaPhys {
  R SoT, SoT1, Re, iRe, sqrt2;
};
template <class Q>
__device__ __forceinline__ SaPhys<double> sa_phys(const Q &P) {
  return SaPhys<double>{P.SoT, 1.0 + P.SoT, P.Re, P.iRe, 1.4142135623730951};
}
template <class Q>
__device__ __forceinline__ SaPhys<float> sa_phys32(const Q &F) {
  return SaPhys<float>{F.SoT, F.SoT1, F.Re, F.iRe, F.sqrt2};
}
__device__ __forceinline__ float over_re(float x, const SaPhys<float> &sp) { return x * sp.iRe; }
__device__ __forceinline__ double over_re(double x, const SaPhys<double> &sp) { return n_div(x, sp.Re); }

// r = nu / (S~ kappa^2 d^2 Re) of the SA destruction term: S~ vanishes in a
// uniform stream, where nu / 0 = inf is the reference's value (capped at 10
// by the caller) and 0 / 0 its NaN, so FP64 divides in full here
__device__ __forceinline__ float sa_r(float nu, float sd2, const SaPhys<float> &sp) {
  return v_div(nu, sd2) * sp.iRe;
}
__device__ __forceinline__ double sa_r(double nu, double sd2, const SaPhys<double> &sp) {
  return nu / (sd2 * sp.Re);
}
// the wall distance with a square in range: the terms of a farther wall vanish
__device__ __forceinline__ float sa_dist(float d) { return d; }
__device__ __forceinline__ double sa_dist(double d) { return r_abs(d) > 1.0e150 ? 1.0e150 : d; }

// Viseddy2mut (Turbulence.cpp:23-30): mu_t = roe fv1 nu, X = nu/(mu/roe)
// clamped at 0, fv1 = X^3/(X^3 + cv1^3).  Here roe fv1, with nul = mu/roe.
__device__ __forceinline__ double sa_roe_fv1(double nu, double roe, double nul) {
#pragma clang fp contract(off)
  double bigx = v_div(nu, nul);
  if (bigx < 0.0) bigx = 0.0;
  const double b2 = bigx * bigx;
  const double fv1 = v_div(b2 * bigx, fma(b2, bigx, SA::cv1three));
  return roe * fv1;
}

// Velocity and temperature of a viscous stencil cell, T = p/(roe Rg)
// (Get_T_ideal_gas).
struct VelT {
  double u, v, w, T;
};
template <int D>
__device__ __forceinline__ VelT vel_t(const Prim<double, D> &q, double Rg) {
  return VelT{q.u, q.v, q.w, v_div(q.p, q.r * Rg)};
}

// Viscous face flux of ComptViscousStress (NS_Solver.cpp:426-581, laminar).
// Stencil of the face between L (low side, the reference's abox, of density
// rL) and Rr: t[0..3] = L+t1, Rr+t1, L-t1, Rr-t1 and, in 3D, t[4..7] the
// same for t2, where t1 < t2 are the two tangential axes.  Gradients: normal
// difference (pfpkesai0) and the four-point tangential difference
// (pfpkesai1), times the cell metric 1/dh (VarReflect with keisa =
// diag(1/dh)); Sutherland mu (:531-533); tau and heat flux (:544-557); output
// A*[0, tau.n, (u.tau+q).n].  With turb set, the SA terms of :534-542: the
// face eddy viscosity mu_t = Viseddy2mut(nu_f, roe_f, mu) joins mu and the
// heat conduction, and mflux receives the face flux of the working variable
// (nu_f + mu/roe_f) (d nu / d n) / sigma * A (the face keisa is the unit
// axis, so the dot product picks the normal derivative).  The quotients by the
// constants 3, Re and Re Pr_t (gama-1) Ma^2 are c_div's, three instructions
// each (as products with the rounded reciprocals the rms error of the normal
// stress grew by 3 %).  FP64.
template <int D>
__device__ __forceinline__ void visc_flux(const VelT &L, const VelT &Rr, double rL, double rR,
                                          const VelT *t, int d, const ViscPhys<double, D> &vp,
                                          double *out, bool turb, double nuL, double nuR,
                                          double *mflux) {
#pragma clang fp contract(off)
  const bool x = d == 0, y = d == 1;
  auto pf1 = [](double a, double b, double c, double e) { return 0.25 * (a + b - c - e); };
  // velocity gradients along x, y, z: the normal difference (pfpkesai0) along
  // d, the tangential ones on the other axes in order (the heat flux is along
  // the normal)
  const double n[3] = {Rr.u - L.u, Rr.v - L.v, Rr.w - L.w};
  const double a[3] = {pf1(t[0].u, t[1].u, t[2].u, t[3].u), pf1(t[0].v, t[1].v, t[2].v, t[3].v),
                       (D == 3) ? pf1(t[0].w, t[1].w, t[2].w, t[3].w) : 0.0};
  double b[3] = {0.0, 0.0, 0.0};
  if constexpr (D == 3) {
    b[0] = pf1(t[4].u, t[5].u, t[6].u, t[7].u);
    b[1] = pf1(t[4].v, t[5].v, t[6].v, t[7].v);
    b[2] = pf1(t[4].w, t[5].w, t[6].w, t[7].w);
  }
  double gx[3], gy[3], gz[3];
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    gx[k] = x ? n[k] : a[k];
    gy[k] = y ? n[k] : (x ? a[k] : b[k]);
    gz[k] = (x || y) ? b[k] : n[k];
  }
  // (x*1 + 0 + 0 is exact; written as a sum so that no per-lane table is built)
  auto axis = [&](double v0, double v1, double v2) {
    return (x ? 1.0 : 0.0) * v0 + (y ? 1.0 : 0.0) * v1 + ((x || y) ? 0.0 : 1.0) * v2;
  };
  const double ih = axis(vp.ih0, vp.ih1, vp.ih2), area = axis(vp.ar0, vp.ar1, vp.ar2);
  const double ftemp = (L.T + Rr.T) * 0.5;
  double mu0 = v_sqrt(ftemp * ftemp * ftemp) * v_div(1.0 + vp.SoT, ftemp + vp.SoT);
  double qk0 = vp.qk * mu0;
  if (turb) {
    const double fvis = (nuL + nuR) * 0.5;
    const double froe = (rL + rR) * 0.5;
    const double nul = v_div(mu0, froe);
    const double rf = sa_roe_fv1(fvis, froe, nul);
    qk0 += c_div(rf * fvis, vp.qkt, vp.iqkt);
    mu0 = fma(rf, fvis, mu0);
    // (1 / segma = 3/2 is exact, segma = 2/3 is not)
    *mflux = (fvis + nul) * ((nuR - nuL) * ih) * (1.0 / SA::segma) * area;
  }
  const double mur = c_div(mu0, vp.Re, vp.iRe);
  // the normal's own term rounded by itself: its rounding is then the same in
  // the sum, and a third of it cancels
  const double dn = x ? gx[0] * vp.ih0 : (y ? gy[1] * vp.ih1 : gz[2] * vp.ih2);
  double divu = y ? gx[0] * vp.ih0 : gy[1] * vp.ih1;
  if (D == 3) divu = fma((x || y) ? gz[2] : gx[0], (x || y) ? vp.ih2 : vp.ih0, divu);
  divu += dn;
  const double tnn = c_div(2.0 * mu0 * (dn - c_div(divu, 3.0, 1.0 / 3.0)), vp.Re, vp.iRe);
  const double txy = mur * fma(gy[0], vp.ih1, gx[1] * vp.ih0);
  const double fu = (L.u + Rr.u) * 0.5, fv = (L.v + Rr.v) * 0.5;
  double t1, t2, work;
  if (D == 2) {
    t1 = x ? tnn : txy;
    t2 = x ? txy : tnn;
    work = fma(fu, t1, fv * t2);
  } else {
    const double txz = mur * fma(gz[0], vp.ih2, gx[2] * vp.ih0);
    const double tyz = mur * fma(gz[1], vp.ih2, gy[2] * vp.ih1);
    t1 = x ? tnn : (y ? txy : txz);
    t2 = x ? txy : (y ? tnn : tyz);
    const double t3 = x ? txz : (y ? tyz : tnn);
    work = fma((L.w + Rr.w) * 0.5, t3, fma(fu, t1, fv * t2));
    out[3] = t3 * area;
  }
  out[0] = 0.0;
  out[1] = t1 * area;
  out[2] = t2 * area;
  out[D == 3 ? 4 : 3] = fma(qk0, (Rr.T - L.T) * ih, work) * area;
}

// The same in 2D FP32 with its fused operations written out, so that the
// form with a known direction (DIR, block tiles) rounds as the one with a
// direction from the face list (DIR = -1).  iL, iR: 1 / (roe Rg) of the two
// cells; tu, tv: the tangential stencil's velocities (its temperatures do
// not enter: the heat flux is along the normal).
template <int DIR>
__device__ __forceinline__ void visc_flux_2d(const Prim<float, 2> &L, const Prim<float, 2> &Rr,
                                             float iL, float iR, const float *tu, const float *tv,
                                             int dir, const ViscPhys<float, 2> &vp, float *out,
                                             bool turb, float nuL, float nuR, float *mflux) {
#pragma clang fp contract(off)
  const bool x = DIR >= 0 ? DIR == 0 : dir == 0;
  const float nu = Rr.u - L.u, nv = Rr.v - L.v;
  const float au = 0.25f * (tu[0] + tu[1] - tu[2] - tu[3]);
  const float av = 0.25f * (tv[0] + tv[1] - tv[2] - tv[3]);
  const float TR = iR * Rr.p;
  const float nT = fmaf(-iL, L.p, TR), sT = fmaf(iL, L.p, TR);   // TR -+ TL
  const float ih = x ? vp.ih0 : vp.ih1, area = x ? vp.ar0 : vp.ar1;
  const float gux = x ? nu : au, guy = x ? au : nu, gvx = x ? nv : av, gvy = x ? av : nv;
  const float ftemp = 0.5f * sT;
  float mu0 = f_sqrt(ftemp * ftemp * ftemp) * ((1.0f + vp.SoT) * f_rcp(fmaf(0.5f, sT, vp.SoT)));
  float qk0 = vp.qk * mu0;
  if (turb) {
    const float fvis = (nuL + nuR) * 0.5f;
    const float froe = (L.r + Rr.r) * 0.5f;
    const float nul = mu0 * f_rcp(froe);
    float bigx = fvis * f_rcp(nul);
    if (bigx < 0.0f) bigx = 0.0f;
    const float b2 = bigx * bigx;
    const float rf = froe * (bigx * b2 * f_rcp(fmaf(bigx, b2, (float)SA::cv1three)));
    qk0 = fmaf(vp.qk, mu0, rf * fvis * vp.iqkt);
    mu0 = fmaf(rf, fvis, mu0);
    *mflux = ((fvis + nul) * ((nuR - nuL) * ih)) * c_rcp((float)SA::segma) * area;
  }
  const float dvy = gvy * vp.ih1;
  const float dv3 = fmaf(gux, vp.ih0, dvy) * c_rcp(3.0f);
  const float dn = x ? gux * vp.ih0 : dvy;
  const float tnn = 2.0f * mu0 * (dn - dv3) * vp.iRe;   // tauxx or tauyy
  const float txy = mu0 * vp.iRe * fmaf(gvx, vp.ih0, guy * vp.ih1);
  const float t1 = x ? tnn : txy, t2 = x ? txy : tnn;
  const float fu = (L.u + Rr.u) * 0.5f, fv = (L.v + Rr.v) * 0.5f;
  out[0] = 0.0f;
  out[1] = t1 * area;
  out[2] = t2 * area;
  out[3] = fmaf(qk0, nT * ih, fmaf(fu, t1, fv * t2)) * area;
}

// The same in 3D (the fused operations are those of the 3D kernels).  t[8]:
// the tangential stencil, t1 then t2.
template <int DIR>
__device__ __forceinline__ void visc_flux_3d(const Prim<float, 3> &L, const Prim<float, 3> &Rr,
                                             float iL, float iR, const Prim<float, 3> *t, int dir,
                                             const ViscPhys<float, 3> &vp, float *out, bool turb,
                                             float nuL, float nuR, float *mflux) {
#pragma clang fp contract(off)
  const int d = DIR >= 0 ? DIR : dir;
  const bool x = d == 0, y = d == 1;
  auto pf = [](float a, float b, float c, float e) { return 0.25f * (a + b - c - e); };
  const float n[3] = {Rr.u - L.u, Rr.v - L.v, Rr.w - L.w};
  const float a[3] = {pf(t[0].u, t[1].u, t[2].u, t[3].u), pf(t[0].v, t[1].v, t[2].v, t[3].v),
                      pf(t[0].w, t[1].w, t[2].w, t[3].w)};
  const float b[3] = {pf(t[4].u, t[5].u, t[6].u, t[7].u), pf(t[4].v, t[5].v, t[6].v, t[7].v),
                      pf(t[4].w, t[5].w, t[6].w, t[7].w)};
  // gradient of component k along x, y, z: the normal difference along d,
  // the tangential ones on the other two axes in order
  float gx[3], gy[3], gz[3];
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    gx[k] = x ? n[k] : a[k];
    gy[k] = y ? n[k] : (x ? a[k] : b[k]);
    gz[k] = (x || y) ? b[k] : n[k];
  }
  const float TL = iL * L.p, TR = iR * Rr.p;
  const float nT = fmaf(iR, Rr.p, -TL), sT = TL + TR;
  // (exact; written as sums so that no per-lane table is built)
  auto axis = [&](float v0, float v1, float v2) {
    if (DIR >= 0) return DIR == 0 ? v0 : (DIR == 1 ? v1 : v2);
    return (x ? 1.0f : 0.0f) * v0 + (y ? 1.0f : 0.0f) * v1 + ((x || y) ? 0.0f : 1.0f) * v2;
  };
  const float ih = axis(vp.ih0, vp.ih1, vp.ih2), area = axis(vp.ar0, vp.ar1, vp.ar2);
  const float ftemp = 0.5f * sT;
  float mu0 = f_sqrt(ftemp * (ftemp * ftemp)) * ((1.0f + vp.SoT) * f_rcp(fmaf(0.5f, sT, vp.SoT)));
  float qk0 = vp.qk * mu0;
  if (turb) {
    const float fvis = (nuL + nuR) * 0.5f;
    const float froe = (L.r + Rr.r) * 0.5f;
    const float ir = f_rcp(froe);
    float bigx = fvis * f_rcp(mu0 * ir);
    if (bigx < 0.0f) bigx = 0.0f;
    const float b2 = bigx * bigx;
    const float rf = froe * (bigx * b2 * f_rcp(fmaf(bigx, b2, (float)SA::cv1three)));
    *mflux = (fmaf(ir, mu0, fvis) * ((nuR - nuL) * ih)) * c_rcp((float)SA::segma) * area;
    qk0 = fmaf(vp.qk, mu0, rf * fvis * vp.iqkt);
    mu0 = fmaf(rf, fvis, mu0);
  }
  const float mur = mu0 * vp.iRe, mu2 = 2.0f * mu0;
  const float dvy = gy[1] * vp.ih1;
  const float dv3 = fmaf(gz[2], vp.ih2, fmaf(gx[0], vp.ih0, dvy)) * c_rcp(3.0f);
  const float dn = x ? gx[0] * vp.ih0 : (y ? dvy : gz[2] * vp.ih2);
  const float tnn = mu2 * (dn - dv3) * vp.iRe;
  const float txy = mur * fmaf(gy[0], vp.ih1, gx[1] * vp.ih0);
  const float txz = mur * fmaf(gx[2], vp.ih0, gz[0] * vp.ih2);
  const float tyz = mur * fmaf(gy[2], vp.ih1, gz[1] * vp.ih2);
  const float t1 = x ? tnn : (y ? txy : txz), t2 = x ? txy : (y ? tnn : tyz);
  const float t3 = x ? txz : (y ? tyz : tnn);
  const float fu = (L.u + Rr.u) * 0.5f, fv = (L.v + Rr.v) * 0.5f, fw = (L.w + Rr.w) * 0.5f;
  const float uv = x ? fmaf(fv, t2, fu * t1) : fmaf(fu, t1, fv * t2);
  out[0] = 0.0f;
  out[1] = t1 * area;
  out[2] = t2 * area;
  out[3] = t3 * area;
  out[4] = fmaf(qk0, nT * ih, fmaf(fw, t3, uv)) * area;
}

// The viscous flux from the stencil cells' states.
template <typename R, int D>
__device__ __forceinline__ void visc_flux_cells(const Prim<R, D> &L, const Prim<R, D> &Rr,
                                                const Prim<R, D> *t, int d,
                                                const ViscPhys<R, D> &vp, R *out, bool turb, R nuL,
                                                R nuR, R *mflux) {
  if constexpr (D == 2 && sizeof(R) == 4) {
    const float tu[4] = {t[0].u, t[1].u, t[2].u, t[3].u}, tv[4] = {t[0].v, t[1].v, t[2].v, t[3].v};
    visc_flux_2d<-1>(L, Rr, f_rcp(L.r * vp.Rg), f_rcp(Rr.r * vp.Rg), tu, tv, d, vp, out, turb, nuL,
                     nuR, mflux);
  } else if constexpr (sizeof(R) == 4) {
    visc_flux_3d<-1>(L, Rr, f_rcp(L.r * vp.Rg), f_rcp(Rr.r * vp.Rg), t, d, vp, out, turb, nuL, nuR,
                     mflux);
  } else {
    VelT vt[(D == 3) ? 8 : 4];
#pragma unroll
    for (int k = 0; k < ((D == 3) ? 8 : 4); ++k) vt[k] = vel_t<D>(t[k], vp.Rg);
    visc_flux<D>(vel_t<D>(L, vp.Rg), vel_t<D>(Rr, vp.Rg), L.r, Rr.r, vt, d, vp, out, turb, nuL, nuR,
                 mflux);
  }
}

// exp, x^6 and x^(1/6) of the SA functions.  FP32: (x^2)^3 and the hardware
// exp2/log2 (v_exp_f32, v_log_f32, ~1 ulp).  FP64: exp is libm's; x^6 is
// (x^2)^3 with the rounding errors of x^2 and x^4 added back; x^(1/6) of
// [6.5e-35, 65/64] (the arguments of sa_fw; below 1.2e-38 the seed would fail)
// takes the FP32 value as the seed (relative error < 1e-5) of two Newton steps
// on y = x^(-1/6), whose error e becomes 7/2 e^2 (1e-5 ->
// 4e-10 -> 5e-19), and returns 1/y.  libm's pow costs ~150 instructions a
// call and the source has three.  Error of fw(r) against 80-bit arithmetic,
// r uniform in [0, 10]: rms 0.9e-16, max 4.4e-16 (pow: 4.5e-16, 6.9e-16);
// in [0, 2]: rms 1.0e-16, max 4.0e-16 (pow: 1.0e-16, 3.7e-16).
template <typename R> __device__ __forceinline__ R r_exp(R x);
template <> __device__ __forceinline__ double r_exp<double>(double x) { return exp(x); }
template <> __device__ __forceinline__ float r_exp<float>(float x) {
  return __builtin_amdgcn_exp2f(x * 1.4426950408889634f);
}
template <typename R> __device__ __forceinline__ R r_pow6(R x);
template <> __device__ __forceinline__ double r_pow6<double>(double x) {
  const double x2 = x * x, e2 = fma(x, x, -x2);
  const double x4 = x2 * x2, e4 = fma(x2, x2, -x4);
  return fma(x4, x2, fma(x4 * e2, 3.0, e4 * x2));
}
template <> __device__ __forceinline__ float r_pow6<float>(float x) {
  const float x2 = x * x;
  return x2 * x2 * x2;
}
template <typename R> __device__ __forceinline__ R r_root6(R x);
template <> __device__ __forceinline__ double r_root6<double>(double x) {
  double y = (double)__builtin_amdgcn_exp2f(__builtin_amdgcn_logf((float)x) * (-1.0f / 6.0f));
#pragma unroll
  for (int k = 0; k < 2; ++k) {
    const double y2 = y * y;
    y = fma(y * (1.0 / 6.0), fma(-x, y2 * y2 * y2, 1.0), y);
  }
  return n_rcp(y);
}
template <> __device__ __forceinline__ float r_root6<float>(float x) {
  return __builtin_amdgcn_exp2f(__builtin_amdgcn_logf(x) * (1.0f / 6.0f));
}

// fw(r) of the SA destruction term: g = r + cw2 (r^6 - r),
// fw = g ((1 + cw3^6) / (g^6 + cw3^6))^(1/6), cw3 = 2.  r is at most 10, but
// has no lower bound where the working variable is negative (set by the
// caller, read from a file, extrapolated): g then grows as r^6 and leaves the
// range of r_root6's FP32 seed.  In FP64 g is held at 1e6, where 64 no longer
// counts beside g^6 and fw has its limit to rounding; once g^6 is infinite
// the formula gives g 0, as pow does.
__device__ __forceinline__ float sa_fw(float r) {
  const float g = r + (float)SA::cw2 * (r_pow6(r) - r);
  return g * r_root6(v_div(65.0f, r_pow6(g) + 64.0f));
}
__device__ __forceinline__ double sa_fw(double r) {
  const double g = r + SA::cw2 * (r_pow6(r) - r);
  const double h = g > 1.0e6 ? 1.0e6 : g;
  const double fw = h * r_root6(v_div(65.0, r_pow6(h) + 64.0));
  return g < 2.3757e51 ? fw : g * 0.0;   // 2^(1024 / 6); NaN stays NaN
}

// ComptMutSource (NS_Solver.cpp:648-808) for one non-solid cell: central
// differences over the face neighbours (nl/nr: working variable, ul..wr:
// velocity, low and high neighbour per axis), vorticity, Sutherland mu,
// fv1/fv2, the modified vorticity S~ (floored at 0.3|Omega|sqrt2), ft2, r, g,
// fw, then advection + production - destruction + cb2 diffusion.  mutf is
// the frozen face-flux term sum(dirsign * mutflux)/V/Re of the step.  The
// frame velocity of the reference is zero here.
template <typename R, int D>
__device__ __forceinline__ R sa_source(R u, R v, R w, R T, R roe, R nu, R sd, const R *nl,
                                       const R *nr, const R *ul, const R *ur, const R *vl,
                                       const R *vr, const R *wl, const R *wr, R ih0, R ih1, R ih2,
                                       const SaPhys<R> &sp, R mutf) {
  sd = sa_dist(sd);
  const R h = R(0.5);
  const R dvisx = ((nr[0] - nl[0]) * h) * ih0;
  const R dvisy = ((nr[1] - nl[1]) * h) * ih1;
  const R dvisz = (D == 3) ? ((nr[2] - nl[2]) * h) * ih2 : R(0);
  const R duy = ((ur[1] - ul[1]) * h) * ih1;
  const R dvx = ((vr[0] - vl[0]) * h) * ih0;
  R duz = R(0), dvz = R(0), dwx = R(0), dwy = R(0);
  if (D == 3) {
    duz = ((ur[2] - ul[2]) * h) * ih2;
    dvz = ((vr[2] - vl[2]) * h) * ih2;
    dwx = ((wr[0] - wl[0]) * h) * ih0;
    dwy = ((wr[1] - wl[1]) * h) * ih1;
  }
  const R ox = R(0.5) * (dwy - dvz), oy = R(0.5) * (duz - dwx), oz = R(0.5) * (dvx - duy);
  const R mu0 = v_sqrt(T * T * T) * v_div(sp.SoT1, T + sp.SoT);
  const R vis0 = v_div(mu0, roe);
  const R bigx = v_div(nu, vis0);
  const R b3 = bigx * bigx * bigx;
  const R fv1 = v_div(b3, b3 + R(SA::cv1three));
  const R fv2 = R(1.0) - v_div(bigx, R(1.0) + bigx * fv1);
  R segdis, vis2d;
  if (r_abs(sd) < R(0.00000001)) {
    segdis = R(1.0);
    vis2d = R(1.0);
  } else {
    segdis = R(SA::kappa) * sd;
    vis2d = v_div(nu, sd);
  }
  segdis *= segdis;
  const R olen = sp.sqrt2 * v_sqrt(ox * ox + oy * oy + oz * oz);
  R bigs = olen + over_re(v_div(nu * fv2, segdis), sp);
  bigs = (R(0.3) * olen < bigs) ? bigs : R(0.3) * olen;
  const R ft2 = R(SA::ct3) * r_exp(-R(SA::ct4) * bigx * bigx);
  R rr = sa_r(nu, bigs * segdis, sp);
  rr = (R(10.0) < rr) ? R(10.0) : rr;
  const R fw = sa_fw(rr);
  R src = -(u * dvisx + v * dvisy + w * dvisz);
  src += R(SA::cb1) * (R(1.0) - ft2) * bigs * nu;
  src -= over_re((R(SA::cw1) * fw - v_div(R(SA::cb1) * ft2, R(SA::kappa * SA::kappa))) * (vis2d * vis2d), sp);
  src += over_re(v_div(R(SA::cb2) * (dvisx * dvisx + dvisy * dvisy + dvisz * dvisz), R(SA::segma)), sp);
  src += mutf;
  return src;
}

// Wall-function fits of Turbulence.cpp:32-55: y+ as a function of the local
// Reynolds number and u+ as a function of y+ (piecewise fits in sqrt and the
// fourth root; FP64 in both modes, as all wall interpolation).
__device__ __forceinline__ double sa_yplus(double re) {
  const double sq = sqrt(re);
  if (re <= 9.0) return 1.002 * sq - 0.001223;
  if (re <= 37.0) return 1.272 * sq - 0.9881 * sqrt(sq) + 0.9054;
  if (re <= 98.0) return 0.2715 * sq + 1.144 * sqrt(sq) + 0.04718 * re;
  if (re <= 250.0) return 0.04921 * sq + 1.576 * sqrt(sq) + 0.05582 * re;
  if (re <= 790.0) return 0.5382 * sq + 0.2478 * sqrt(sq) + 0.04593 * re;
  if (re <= 2800.0) return 1.105 * sq - 1.782 * sqrt(sq) + 0.03933 * re;
  return 2.643 * sq - 10.52 * sqrt(sq) + 0.03207 * re;
}

__device__ __forceinline__ double sa_uplus(double y) {
  if (y < 3.0) return y;
  const double lg = log(y), sq = sqrt(y), qu = sqrt(sq);
  if (y < 8.5) return -6.645 * lg + 25.59 * sq - 21.6 * qu - 1.864 * y;
  if (y < 50.0) return 12.04 * lg - 4.079 * sq - 4.504 * qu + 0.1715 * y;
  if (y < 300.0) return 3.031 * lg - 0.6252 * sq + 2.639 * qu + 0.007553 * y;
  if (y < 1000.0) return -3.535 * lg - 1.104 * sq + 13.89 * qu + 0.004011 * y;
  return 16.66 * lg + 1.408 * sq - 23.82 * qu - 0.002909 * y;
}

}  // namespace ibg
