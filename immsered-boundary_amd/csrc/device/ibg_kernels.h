// ibg_kernels.h — HIP kernels of the residual engine (gfx950).
//
// Conventions: R is the arithmetic type of the flux kernels (double in the
// plain mode, float in the mixed mode); D is 2 or 3; NV = D+2 values per
// cell.  Every ghost fill, the CFL time step, the wall force and the
// conserved state are FP64 in both modes.
#pragma once
#include <hip/hip_runtime.h>

#include "ibg_block.h"
#include "ibg_common.h"
#include "ibg_flux.h"
#include "ibg_mlp.h"

#include <type_traits>

namespace ibg {

constexpr int kTile = 256;   // cells per workgroup of the tiled kernels (max)

__device__ __forceinline__ TileInfo tile_info(const TileInfo *tiles, int t) {
  const auto *p = uni(tiles) + t;
  return TileInfo{p->cell0, p->ncell, p->face0, p->nface, p->blk, p->halo0, 0, 0};
}

// ------------------------------------------------------------ pack access
template <typename R, int D>
__device__ __forceinline__ Prim<R, D> pload(const Pack<R, D> &W, int c) {
  const typename V4<R>::T q = W.a[c];
  Prim<R, D> o;
  o.r = q.x; o.u = q.y; o.v = q.z;
  if (D == 2) { o.w = R(0); o.p = q.w; }
  else { o.w = q.w; o.p = W.e[c]; }
  return o;
}

// the records from cell c0 on
template <typename R, int D>
__device__ __forceinline__ Pack<R, D> rebase(const Pack<R, D> &W, int c0) {
  return Pack<R, D>{W.a + c0, D == 3 ? W.e + c0 : W.e};
}

// velocity of cell c (the 4-vector only; w = 0 in 2D)
template <typename R, int D>
__device__ __forceinline__ void uvw_load(const Pack<R, D> &W, int c, R &u, R &v, R &w) {
  const typename V4<R>::T q = W.a[c];
  u = q.y; v = q.z;
  w = (D == 3) ? q.w : R(0);
}

template <typename R, int D>
__device__ __forceinline__ void pstore(const Pack<R, D> &W, int c, R r, R u, R v, R w, R p) {
  typename V4<R>::T q;
  q.x = r; q.y = u; q.z = v;
  if (D == 2) { q.w = p; }
  else { q.w = w; W.e[c] = p; }
  W.a[c] = q;
}

// NV-value records (conserved state, residuals): values 0..3 in a, 4 in e
template <typename R, int D>
__device__ __forceinline__ void vload(const Pack<R, D> &P, int c, R *o) {
  const typename V4<R>::T q = P.a[c];
  o[0] = q.x; o[1] = q.y; o[2] = q.z; o[3] = q.w;
  if (D == 3) o[4] = P.e[c];
}

template <typename R, int D>
__device__ __forceinline__ void vstore(const Pack<R, D> &P, int c, const R *v) {
  typename V4<R>::T q;
  q.x = v[0]; q.y = v[1]; q.z = v[2]; q.w = v[3];
  P.a[c] = q;
  if (D == 3) P.e[c] = v[4];
}

// Ghost-fill write: the FP64 master and every stencil copy (see StateOut).
template <int D>
__device__ __forceinline__ void put_all(const StateOut<D> &o, int c, double r, double u, double v,
                                        double w, double p) {
  pstore<double, D>(o.m, c, r, u, v, w, p);
  if (o.nd > 0) pstore<double, D>(o.d1, c, r, u, v, w, p);
  if (o.nd > 1) pstore<double, D>(o.d2, c, r, u, v, w, p);
  if (o.nf > 0) pstore<float, D>(o.f0, c, (float)r, (float)u, (float)v, (float)w, (float)p);
  if (o.nf > 1) pstore<float, D>(o.f1, c, (float)r, (float)u, (float)v, (float)w, (float)p);
  if (o.nf > 2) pstore<float, D>(o.f2, c, (float)r, (float)u, (float)v, (float)w, (float)p);
}

template <int D>
__device__ __forceinline__ void put_nu(const StateOut<D> &o, int c, double nu) {
  if (!o.nm) return;
  o.nm[c] = nu;
  if (o.nd > 0) o.nd1[c] = nu;
  if (o.nd > 1) o.nd2[c] = nu;
  if (o.nf > 0) o.nf0[c] = (float)nu;
  if (o.nf > 1) o.nf1[c] = (float)nu;
  if (o.nf > 2) o.nf2[c] = (float)nu;
}

// error word: ((cell << 16) | code), the smallest cell wins
__device__ __forceinline__ void report_error(unsigned long long *err, int cell, int code) {
  unsigned long long v = ((unsigned long long)(unsigned)cell << 16) | (unsigned)code;
  atomicMin(err, v);
}

// ------------------------------------------------------------ stage kernel
// ----------------------------------------- viscous flux + step preparation
template <typename R, int D>
struct ViscArgs {
  const TileInfo *tiles;
  const int4 *tst;           // L, R from .y, .z
  const int4 *tvs;           // [nface][D-1] tangential stencil
  const int8_t *tdir;
  const int *halo;           // halo lists of the block tiles
  const uint16_t *slots;
  const BlkInfo *blk;
  const DevPhys *phys;
  const Flow32 *flow;        // per block (FP32)
  Pack<R, D> W;              // step-start stencil state
  Pack<R, D> Rv;
  const R *nu;               // SA working variable (turb)
  R *mutf;                   // [Nn] frozen face-flux term (turb)
  int viscous, turb;
  const unsigned long long *err;
  // optional coarse/fine balance: tile face -> entry of rbalv (-1: none);
  // rbalv NULL when the balance is off
  const int *tmod;
  const R *rbalv;
};

template <typename R, int D>
__device__ __forceinline__ ViscPhys<R, D> visc_phys(const BlkInfo *blks, const DevPhys *phys,
                                                    const Flow32 *flow, int blk) {
  ViscPhys<R, D> vp;
  if constexpr (sizeof(R) == 4) {
    const auto &F = uni(flow)[blk];
    vp.Rg = F.Rg; vp.iRe = F.iRe; vp.qk = F.qk; vp.SoT = F.SoT;
    vp.ih0 = F.invh[0]; vp.ih1 = F.invh[1]; vp.ih2 = F.invh[2];
    vp.ar0 = F.area[0]; vp.ar1 = F.area[1]; vp.ar2 = F.area[2];
    vp.iqkt = F.iqkt;
  } else {
    const auto &bi = uni(blks)[blk];
    const auto &P = uni(phys)[bi.case_id];
    vp.Rg = P.Rg; vp.iRe = P.iRe; vp.qk = P.qk; vp.SoT = P.SoT;
    vp.ih0 = bi.invh[0]; vp.ih1 = bi.invh[1]; vp.ih2 = bi.invh[2];
    vp.ar0 = bi.area[0]; vp.ar1 = bi.area[1]; vp.ar2 = bi.area[2];
    vp.iqkt = P.iqkt;
    vp.Re = P.Re; vp.qkt = P.qkt_den;
  }
  return vp;
}
template <typename R, int D>
__device__ __forceinline__ ViscPhys<R, D> visc_phys(const ViscArgs<R, D> &a, int blk) {
  return visc_phys<R, D>(a.blk, a.phys, a.flow, blk);
}

// The FP32 constants of block b (see Flow32).
__global__ void k_flow32(int nblk, const BlkInfo *blk, const DevPhys *phys, Flow32 *out) {
  const int b = blockIdx.x * blockDim.x + threadIdx.x;
  if (b >= nblk) return;
  const BlkInfo &B = blk[b];
  const DevPhys &P = phys[B.case_id];
  Flow32 F;
  for (int d = 0; d < 3; ++d) { F.area[d] = (float)B.area[d]; F.invh[d] = (float)B.invh[d]; }
  const PhysR<float> ph = phys_r<float>(P);
  F.gama = ph.gama; F.Rg = ph.Rg; F.Cv = ph.Cv; F.Ma = ph.Ma;
  F.gm1 = ph.gm1; F.ig1 = ph.ig1; F.iRg = ph.iRg; F.cpR = ph.cpR;
  F.SoT = (float)P.SoT; F.SoT1 = 1.0f + F.SoT;
  F.Re = (float)P.Re; F.iRe = f_rcp(F.Re);
  F.qk = (float)P.qk; F.iqkt = f_rcp((float)P.qkt_den);
  F.sqrt2 = v_sqrt(2.0f);
  F.pad = 0.0f;
  out[b] = F;
}

// The viscous flux (and, with the SA closure, the working variable's face
// flux mf) of tile face k (an index into tst / tvs / tdir).
template <typename R, int D>
__device__ __forceinline__ void visc_face(const ViscArgs<R, D> &a, const ViscPhys<R, D> &vp, int k,
                                          R *out, R &mf) {
  const int4 st = a.tst[k];
  const int dir = a.tdir[k];
  const Prim<R, D> L = pload<R, D>(a.W, st.y);
  const Prim<R, D> Rr = pload<R, D>(a.W, st.z);
  Prim<R, D> t[(D == 3) ? 8 : 4];
  const int4 v0 = a.tvs[(size_t)k * (D - 1)];
  t[0] = pload<R, D>(a.W, v0.x); t[1] = pload<R, D>(a.W, v0.y);
  t[2] = pload<R, D>(a.W, v0.z); t[3] = pload<R, D>(a.W, v0.w);
  if (D == 3) {
    const int4 v1 = a.tvs[(size_t)k * (D - 1) + 1];
    t[4 % ((D == 3) ? 8 : 4)] = pload<R, D>(a.W, v1.x);
    t[5 % ((D == 3) ? 8 : 4)] = pload<R, D>(a.W, v1.y);
    t[6 % ((D == 3) ? 8 : 4)] = pload<R, D>(a.W, v1.z);
    t[7 % ((D == 3) ? 8 : 4)] = pload<R, D>(a.W, v1.w);
  }
  mf = R(0);
  if (a.turb)
    visc_flux_cells<R, D>(L, Rr, t, dir, vp, out, true, a.nu[st.y], a.nu[st.z], &mf);
  else
    visc_flux_cells<R, D>(L, Rr, t, dir, vp, out, false, R(0), R(0), &mf);
}

// Once per step (ComptViscousStress NS_Solver.cpp:365-629 is frozen across
// the stages, NS_Solver.H:669-699): viscous fluxes of the tile faces into
// LDS, then per cell Rv = sum_d (Fv_hi - Fv_lo).  With the SA closure the
// face flux of the working variable (mutflux, :534-542) is reduced the same
// way into sum_d (mutflux_hi - mutflux_lo) / V / Re (:791-800).
// halt: an LDS flag that thread 0 sets from herr (the error word, loaded at
// kernel start) just before the face phase's barrier and that every thread
// tests after it: a halted workgroup writes nothing.
template <typename R, int D>
__device__ __forceinline__ void visc_prep_tile(const ViscArgs<R, D> &a, const TileInfo &ti,
                                               unsigned char *smem_raw, int *halt, bool herr) {
  constexpr int NV = D + 2;
  using V = typename V4<R>::T;
  V *fl4 = reinterpret_cast<V *>(smem_raw);
  R *fl1 = reinterpret_cast<R *>(smem_raw + sizeof(V) * (size_t)ti.nface);
  R *mfl = reinterpret_cast<R *>(smem_raw + (sizeof(V) + (D == 3 ? sizeof(R) : 0)) * (size_t)ti.nface);
  auto &bi = uni(a.blk)[ti.blk];
  auto &P = uni(a.phys)[bi.case_id];
  if (a.viscous) {
    const ViscPhys<R, D> vp = visc_phys<R, D>(a, ti.blk);
    for (int f = threadIdx.x; f < ti.nface; f += blockDim.x) {
      R out[NV];
      R mf;
      visc_face<R, D>(a, vp, ti.face0 + f, out, mf);
      if (a.rbalv) {
        // a coarse/fine face of the optional balance: its balanced flux
        const int q = a.tmod[ti.face0 + f];
        if (q >= 0)
          for (int v = 0; v < NV; ++v) out[v] = a.rbalv[(size_t)q * NV + v];
      }
      V o;
      o.x = out[0]; o.y = out[1]; o.z = out[2]; o.w = out[3];
      fl4[f] = o;
      if (D == 3) fl1[f] = out[4];
      if (a.turb) mfl[f] = mf;
    }
  }
  if (threadIdx.x == 0) *halt = herr ? 1 : 0;
  __syncthreads();
  if (*halt) return;
  const int i = threadIdx.x;
  if (i >= ti.ncell) return;   // no barrier follows in this function
  const int c = ti.cell0 + i;
  double s[NV];
#pragma unroll
  for (int k = 0; k < NV; ++k) s[k] = 0.0;
  double tot = 0.0;
  if (a.viscous) {
    int sl[2 * D];
    if (D == 2) {
      const ushort4 s4 = *reinterpret_cast<const ushort4 *>(a.slots + (size_t)c * 4);
      sl[0] = s4.x; sl[1] = s4.y; sl[2] = s4.z; sl[3] = s4.w;
    } else {
#pragma unroll
      for (int q = 0; q < 2 * D; ++q) sl[q] = a.slots[(size_t)c * 2 * D + q];
    }
#pragma unroll
    for (int d = 0; d < D; ++d) {
      const int lo = sl[2 * d], hi = sl[2 * d + 1];
      const V flo = fl4[lo], fhi = fl4[hi];
      s[0] += (double)fhi.x - (double)flo.x;
      s[1] += (double)fhi.y - (double)flo.y;
      s[2] += (double)fhi.z - (double)flo.z;
      s[3] += (double)fhi.w - (double)flo.w;
      if (D == 3) s[4] += (double)fl1[hi] - (double)fl1[lo];
      if (a.turb) {
        // total_face_flux += dirsign[f0] * mutflux, dirsign = {-1, +1}
        tot += -(double)mfl[lo];
        tot += (double)mfl[hi];
      }
    }
  }
  R rv[NV];
#pragma unroll
  for (int k = 0; k < NV; ++k) rv[k] = (R)s[k];
  vstore<R, D>(a.Rv, c, rv);
  if (a.turb) a.mutf[c] = (R)n_div(n_div(tot, bi.vol), P.Re);
}

// ---------------------------------------------------------- block tiles
// The LDS of a block tile (ibg_block.h).
// n 4-vectors in LDS: FP32 whole, FP64 as two planes of 16-byte halves (a
// 32-byte stride would leave every second group of four banks idle).
template <typename R>
struct LdsVec {
  using V = typename V4<R>::T;
  V *q;
  __device__ __forceinline__ V operator[](int p) const { return q[p]; }
  __device__ __forceinline__ void put(int p, const V &v) const { q[p] = v; }
  __device__ __forceinline__ LdsVec from(int p) const { return LdsVec{q + p}; }
};
template <>
struct LdsVec<double> {
  using V = D4;
  double2 *a, *b;
  __device__ __forceinline__ D4 operator[](int p) const {
    const double2 x = a[p], y = b[p];
    return D4{x.x, x.y, y.x, y.y};
  }
  __device__ __forceinline__ void put(int p, const D4 &v) const {
    a[p] = make_double2(v.x, v.y);
    b[p] = make_double2(v.z, v.w);
  }
  __device__ __forceinline__ LdsVec from(int p) const { return LdsVec{a + p, b + p}; }
};
template <typename R>
__device__ __forceinline__ LdsVec<R> lds_vec(unsigned char *smem, int n) {
  if constexpr (sizeof(R) == 4) {
    return LdsVec<R>{reinterpret_cast<typename V4<R>::T *>(smem)};
  } else {
    double2 *h = reinterpret_cast<double2 *>(smem);
    return LdsVec<R>{h, h + n};
  }
}
template <typename R>
struct BlockLds {
  LdsVec<R> fx, fy;             // fluxes of the x and y faces
  LdsVec<R> S;                  // states of the box
  R *nu, *T;                    // working variable (SA); temperature for the
                                // viscous flux (FP64)
};
template <typename R>
__device__ __forceinline__ BlockLds<R> block_lds(unsigned char *smem, bool turb) {
  BlockLds<R> b;
  b.fx = lds_vec<R>(smem, kFluxSlots);
  b.fy = b.fx.from(kFxSlots);
  unsigned char *st = smem + blk_state_offset(sizeof(R));
  b.S = lds_vec<R>(st, kBoxCells);
  b.nu = reinterpret_cast<R *>(st + 4 * sizeof(R) * kBoxCells);
  b.T = b.nu + (turb ? kBoxCells : 0);
  return b;
}
template <typename R>
__device__ __forceinline__ Prim<R, 2> box_prim(const BlockLds<R> &b, int p) {
  const typename V4<R>::T q = b.S[p];
  return Prim<R, 2>{q.x, q.y, q.z, R(0), q.w};
}

// The square and its first nhalo halo entries into LDS (256 threads; the
// caller syncs).  p0: this thread's cell in the box.  kT: BlockLds::T too.
template <typename R, bool kT>
__device__ __forceinline__ void block_load(const Pack<R, 2> &W, const R *nu, bool turb,
                                           const int *halo, const TileInfo &ti, int nhalo, R Rg,
                                           const BlockLds<R> &b, int p0) {
  // arrays from the tile's first entry on: a uniform base and a 32-bit offset
  const unsigned i = threadIdx.x;
  int hc = 0;
  if ((int)i < nhalo) hc = (halo + ti.halo0)[i];
  auto put = [&](int p, const typename V4<R>::T &q, R n) {
    if constexpr (kT) b.T[p] = v_div(q.w, q.x * Rg);
    b.S.put(p, q);
    if (turb) b.nu[p] = n;
  };
  const typename V4<R>::T q = (W.a + ti.cell0)[i];
  const R n = turb ? (nu + ti.cell0)[i] : R(0);
  if ((int)i < nhalo) {
    const typename V4<R>::T qh = W.a[hc];
    const R nh = turb ? nu[hc] : R(0);
    put(halo_pos((int)i), qh, nh);
  }
  put(p0, q, n);
}

// The faces of a block tile, f(direction or -1, direction, x, y of the
// high-side cell): the low faces of this thread's cell (x, y), then the
// last column's x and the last row's y faces, half a wave together.  That
// wave is another one from workgroup to workgroup, so that the third pass
// does not always fall on the same SIMD.
template <class F>
__device__ __forceinline__ void block_faces(int x, int y, F f) {
  f(std::integral_constant<int, 0>(), 0, x, y);
  // (no overlap of the two: it would cost the registers of both)
  asm volatile("" ::: "memory");
  f(std::integral_constant<int, 1>(), 1, x, y);
  asm volatile("" ::: "memory");
  const int l = threadIdx.x & 63;
  if (((threadIdx.x >> 6) ^ blockIdx.x) & 3 || l >= 2 * kBlkN) return;
  const int dir = l >> 4, t = l & (kBlkN - 1);
  f(std::integral_constant<int, -1>(), dir, dir == 0 ? kBlkN : t, dir == 0 ? t : kBlkN);
}
// the same with the box position of the high-side cell, p that of this thread's
template <class F>
__device__ __forceinline__ void block_faces(int p, F f) {
  block_faces(0, 0, [&](auto dc, int dir, int x, int y) {
    f(dc, dir, decltype(dc)::value >= 0 ? p : box_pos(x, y));
  });
}
// box position of this thread's cell
__device__ __forceinline__ int block_cell() {
  int x, y;
  blk_xy(threadIdx.x, x, y);
  return box_pos(x, y);
}

// FP64 viscous fluxes of the faces into LDS, the working variable's face flux
// in the mass slot (the viscous mass flux is zero).  p: this thread's cell.
template <typename R>
__device__ __forceinline__ void block_visc_faces(const BlockLds<R> &b, const ViscPhys<R, 2> &vp,
                                                 bool turb, int p0) {
  block_faces(p0, [&](auto dc, int dir, int p) {
    constexpr int d = decltype(dc)::value;
    const int st = dir == 0 ? 1 : kBoxP, tt = dir == 0 ? kBoxP : 1;
    const int l = p - st;
    R out[4], mf = R(0);
    const R nl = turb ? b.nu[l] : R(0), nr = turb ? b.nu[p] : R(0);
    const int tp[4] = {l + tt, p + tt, l - tt, p - tt};
    auto cell = [&](int q) {
      const typename V4<R>::T s = b.S[q];
      return VelT{s.y, s.z, 0.0, b.T[q]};
    };
    const VelT t[4] = {cell(tp[0]), cell(tp[1]), cell(tp[2]), cell(tp[3])};
    visc_flux<2>(cell(l), cell(p), b.S[l].x, b.S[p].x, t, dir, vp, out, turb, nl, nr, &mf);
    typename V4<R>::T o;
    o.x = mf; o.y = out[1]; o.z = out[2]; o.w = out[3];
    b.fx.put(p - box_pos(0, 0) + (dir == 0 ? 0 : kFxSlots), o);
  });
}

// Rv and the working variable's face term of this thread's cell from the
// face fluxes in LDS.
template <typename R, class B, class Q>
__device__ __forceinline__ void block_visc_cell(const ViscArgs<R, 2> &a, const TileInfo &ti, B &bi,
                                                Q &P, const BlockLds<R> &b, int p) {
  using V = typename V4<R>::T;
  const unsigned c = threadIdx.x;
  double s[4] = {0.0, 0.0, 0.0, 0.0}, tot = 0.0;
  if (a.viscous) {
    const int k = p - box_pos(0, 0);
#pragma unroll
    for (int d = 0; d < 2; ++d) {
      const V lo = d == 0 ? b.fx[k] : b.fy[k], hi = d == 0 ? b.fx[k + 1] : b.fy[k + kBoxP];
      s[1] += (double)hi.y - (double)lo.y;
      s[2] += (double)hi.z - (double)lo.z;
      s[3] += (double)hi.w - (double)lo.w;
      if (a.turb) {
        tot += -(double)lo.x;
        tot += (double)hi.x;
      }
    }
  }
  const R rv[4] = {(R)s[0], (R)s[1], (R)s[2], (R)s[3]};
  vstore<R, 2>(rebase(a.Rv, ti.cell0), c, rv);
  if (a.turb) (a.mutf + ti.cell0)[c] = (R)n_div(n_div(tot, bi.vol), P.Re);
}

// The FP32 viscous pass of a block tile up to the fluxes in LDS (layout:
// ibg_block.h).  (x, y): this thread's cell.  The halo's first layer only.
__device__ __forceinline__ void block_visc_faces32(const ViscArgs<float, 2> &a, const TileInfo &ti,
                                                   unsigned char *smem, const BlockLds<float> &b,
                                                   int x, int y) {
  float2 *uv = reinterpret_cast<float2 *>(smem + 16 * (size_t)kFluxSlots);
  float2 *rp = uv + kViscCells, *in = rp + kViscCells;
  const ViscPhys<float, 2> vp = visc_phys<float, 2>(a, ti.blk);
  const unsigned i = threadIdx.x;
  int hc = 0;
  if ((int)i < kHaloC) hc = (a.halo + ti.halo0)[i];
  auto put = [&](int p, const F4 &q, float n) {
    uv[p] = make_float2(q.y, q.z);
    rp[p] = make_float2(q.x, q.w);
    in[p] = make_float2(f_rcp(q.x * vp.Rg), n);
  };
  const F4 q = (a.W.a + ti.cell0)[i];
  const float n = a.turb ? (a.nu + ti.cell0)[i] : 0.0f;
  if ((int)i < kHaloC) {
    const F4 qh = a.W.a[hc];
    const float nh = a.turb ? a.nu[hc] : 0.0f;
    int hx, hy;
    halo_xy((int)i, hx, hy);
    put(visc_pos(hx, hy), qh, nh);
  }
  const int p0 = visc_pos(x, y);
  put(p0, q, n);
  __syncthreads();
  block_faces(x, y, [&](auto dc, int dir, int fx, int fy) {
    constexpr int d = decltype(dc)::value;
    const int p = d >= 0 ? p0 : visc_pos(fx, fy);
    const int st = dir == 0 ? 1 : kViscP, tt = dir == 0 ? kViscP : 1;
    const int l = p - st;
    const int tp[4] = {l + tt, p + tt, l - tt, p - tt};
    float tu[4], tv[4], out[4], mf = 0.0f;
#pragma unroll
    for (int k = 0; k < 4; ++k) { const float2 v = uv[tp[k]]; tu[k] = v.x; tv[k] = v.y; }
    const float2 vl = uv[l], vr = uv[p], sl = rp[l], sr = rp[p], il = in[l], ir = in[p];
    visc_flux_2d<d>(Prim<float, 2>{sl.x, vl.x, vl.y, 0.0f, sl.y},
                    Prim<float, 2>{sr.x, vr.x, vr.y, 0.0f, sr.y}, il.x, ir.x, tu, tv, dir, vp, out,
                    a.turb, il.y, ir.y, &mf);
    b.fx.put(fy * kBoxP + fx + (dir == 0 ? 0 : kFxSlots), F4{mf, out[1], out[2], out[3]});
  });
}

// The viscous pass of a block tile (visc_prep_tile's work).
template <typename R>
__device__ __forceinline__ void visc_prep_block(const ViscArgs<R, 2> &a, const TileInfo &ti,
                                                unsigned char *smem_raw, int *halt, bool herr) {
  auto &bi = uni(a.blk)[ti.blk];
  auto &P = uni(a.phys)[bi.case_id];
  const BlockLds<R> b = block_lds<R>(smem_raw, a.turb);
  int x, y;
  blk_xy(threadIdx.x, x, y);
  const int p = box_pos(x, y);
  if (a.viscous) {
    if constexpr (sizeof(R) == 4) {
      block_visc_faces32(a, ti, smem_raw, b, x, y);
    } else {
      block_load<R, true>(a.W, a.nu, a.turb, a.halo, ti, kHaloC, P.Rg, b, p);
      __syncthreads();
      block_visc_faces<R>(b, visc_phys<R, 2>(a, ti.blk), a.turb, p);
    }
  }
  if (threadIdx.x == 0) *halt = herr ? 1 : 0;
  __syncthreads();
  if (*halt) return;
  block_visc_cell<R>(a, ti, bi, P, b, p);
}

// ---- 3D
template <typename R>
struct Block3Lds {
  LdsVec<R> F;            // fluxes of one direction: values 0..3
  R *Fe;                  // value 4
  LdsVec<R> S;            // states (roe, u, v, w)
  R *e, *nu;              // pressure (viscous pass, FP64: temperature); SA
};
template <typename R>
__device__ __forceinline__ Block3Lds<R> block3_lds(unsigned char *smem, int cells) {
  Block3Lds<R> b;
  b.F = lds_vec<R>(smem, kFlux3);
  b.Fe = reinterpret_cast<R *>(smem + 4 * sizeof(R) * kFlux3);
  unsigned char *st = smem + blk3_state_offset(sizeof(R));
  b.S = lds_vec<R>(st, cells);
  b.e = reinterpret_cast<R *>(st + 4 * sizeof(R) * cells);
  b.nu = b.e + cells;
  return b;
}
template <typename R>
__device__ __forceinline__ Prim<R, 3> box3_prim(const Block3Lds<R> &b, int p) {
  const typename V4<R>::T q = b.S[p];
  return Prim<R, 3>{q.x, q.y, q.z, q.w, b.e[p]};
}

// The block and its halo into LDS (the caller syncs).  VISC: layer 1 and the
// edges into the viscous pass's box; otherwise layers 1 and 2.
template <typename R, bool VISC>
__device__ __forceinline__ void block3_load(const Pack<R, 3> &W, const R *nu, bool turb,
                                            const int *halo, const TileInfo &ti, R Rg,
                                            const Block3Lds<R> &b) {
  const int i = threadIdx.x;
  // second entry of this thread: an edge (80 of them) or a cell of layer 2
  const bool has1 = !VISC || i < kHalo3E - kHalo3L1;
  const int h1 = VISC ? kHalo3L1 + i : kHalo3E + i;
  const int c0 = halo[ti.halo0 + i];
  const int c1 = has1 ? halo[ti.halo0 + h1] : 0;
  auto put = [&](int x, int y, int z, const typename V4<R>::T &q, R p, bool n, R nv) {
    const int k = VISC ? vbox3_pos(x, y, z) : box3_pos(x, y, z);
    b.S.put(k, q);
    b.e[k] = (VISC && sizeof(R) == 8) ? v_div(p, q.x * Rg) : p;
    if (n) b.nu[k] = nv;
  };
  const int c = ti.cell0 + i;
  const typename V4<R>::T q = W.a[c], q0 = W.a[c0];
  const R p = W.e[c], p0 = W.e[c0];
  const R n = turb ? nu[c] : R(0), n0 = turb ? nu[c0] : R(0);
  int x, y, z;
  if (has1) {
    const typename V4<R>::T q1 = W.a[c1];
    const R p1 = W.e[c1];
    halo3_xyz(h1, x, y, z);
    put(x, y, z, q1, p1, false, R(0));
  }
  halo3_xyz(i, x, y, z);
  put(x, y, z, q0, p0, turb, n0);
  blk_xyz(i, x, y, z);
  put(x, y, z, q, p, turb, n);
}

// The sums are formed here: left to the compiler, the subtractions of all
// three directions move behind the last one and their operands, sixty
// registers in FP64, are held until then (168 registers and 8 spilled; with
// the sums formed here 145: k_stage 221 -> 212 us).
__device__ __forceinline__ void sum_now(double (&s)[5]) {
#pragma unroll
  for (int k = 0; k < 5; ++k) asm volatile("" : "+v"(s[k]));
}

// The faces of a block in direction d, f(x, y, z of the high-side cell): the
// low face of this thread's cell, then the last layer's high faces by one
// wave, another one from workgroup to workgroup and direction to direction.
// The cell's position serves every phase: k_stage 122 -> 118 us in FP32, 229
// -> 221 in FP64, against positions formed anew in each.
template <int d, class F>
__device__ __forceinline__ void block3_faces(int x, int y, int z, F f) {
  f(x, y, z);
  asm volatile("" ::: "memory");   // (no overlap of the two, as in block_faces)
  const int e = threadIdx.x & 63, u = e & 7, v = e >> 3;
  if (((threadIdx.x >> 6) ^ (blockIdx.x + d)) & 3 || (d < 2 && e >= 32)) return;
  f(d == 0 ? kB3X : u, d == 0 ? u : (d == 1 ? kB3Y : v), d == 2 ? kB3Z : v);
}

// The viscous pass of a 3D block tile (visc_prep_tile's work), one direction
// at a time.
template <typename R>
__device__ __forceinline__ void visc_prep_block3(const ViscArgs<R, 3> &a, const TileInfo &ti,
                                                 unsigned char *smem_raw, int *halt, bool herr) {
  using V = typename V4<R>::T;
  auto &bi = uni(a.blk)[ti.blk];
  auto &P = uni(a.phys)[bi.case_id];
  const Block3Lds<R> b = block3_lds<R>(smem_raw, kVBox3Cells);
  if (threadIdx.x == 0) *halt = herr ? 1 : 0;
  int cx, cy, cz;
  blk_xyz(threadIdx.x, cx, cy, cz);
  double s[5] = {0.0, 0.0, 0.0, 0.0, 0.0}, tot = 0.0;
  if (a.viscous) {
    block3_load<R, true>(a.W, a.nu, a.turb, a.halo, ti, (R)P.Rg, b);
    const ViscPhys<R, 3> vp = visc_phys<R, 3>(a, ti.blk);
    __syncthreads();
    auto direction = [&](auto dc) {
      constexpr int d = decltype(dc)::value;
      constexpr int st[3] = {1, kVBox3P, kVBox3Plane};
      constexpr int sn = st[d], s1 = st[d == 0 ? 1 : 0], s2 = st[d == 2 ? 1 : 2];
      block3_faces<d>(cx, cy, cz, [&](int x, int y, int z) {
        const int p = vbox3_pos(x, y, z), l = p - sn;
        const int tp[8] = {l + s1, p + s1, l - s1, p - s1, l + s2, p + s2, l - s2, p - s2};
        const R nl = a.turb ? b.nu[l] : R(0), nr = a.turb ? b.nu[p] : R(0);
        R out[5], mf = R(0);
        if constexpr (sizeof(R) == 4) {
          Prim<R, 3> t[8];
#pragma unroll
          for (int k = 0; k < 8; ++k) t[k] = box3_prim<R>(b, tp[k]);
          const Prim<R, 3> L = box3_prim<R>(b, l), Rr = box3_prim<R>(b, p);
          visc_flux_3d<d>(L, Rr, f_rcp(L.r * vp.Rg), f_rcp(Rr.r * vp.Rg), t, d, vp, out, a.turb, nl, nr, &mf);
        } else {
          auto cell = [&](int q) {
            const V v = b.S[q];
            return VelT{v.y, v.z, v.w, b.e[q]};
          };
          VelT t[8];
#pragma unroll
          for (int k = 0; k < 8; ++k) t[k] = cell(tp[k]);
          visc_flux<3>(cell(l), cell(p), b.S[l].x, b.S[p].x, t, d, vp, out, a.turb, nl, nr, &mf);
        }
        V o;
        o.x = mf; o.y = out[1]; o.z = out[2]; o.w = out[3];
        const int k = flux3_slot(d, x, y, z);
        b.F.put(k, o);
        b.Fe[k] = out[4];
      });
      __syncthreads();
      const int k = flux3_slot(d, cx, cy, cz), h = flux3_slot(d, cx + (d == 0), cy + (d == 1), cz + (d == 2));
      const V lo = b.F[k], hi = b.F[h];
      s[1] += (double)hi.y - (double)lo.y;
      s[2] += (double)hi.z - (double)lo.z;
      s[3] += (double)hi.w - (double)lo.w;
      s[4] += (double)b.Fe[h] - (double)b.Fe[k];
      if (a.turb) {
        tot += -(double)lo.x;
        tot += (double)hi.x;
      }
      sum_now(s);
      asm volatile("" : "+v"(tot));
      if (d < 2) __syncthreads();   // the next direction rewrites the fluxes
    };
    direction(std::integral_constant<int, 0>());
    direction(std::integral_constant<int, 1>());
    direction(std::integral_constant<int, 2>());
  } else {
    __syncthreads();
  }
  if (*halt) return;   // uniform: written before the barriers
  const int c = ti.cell0 + threadIdx.x;
  const R rv[5] = {(R)s[0], (R)s[1], (R)s[2], (R)s[3], (R)s[4]};
  vstore<R, 3>(a.Rv, c, rv);
  if (a.turb) a.mutf[c] = (R)n_div(n_div(tot, bi.vol), P.Re);
}

// (waves per SIMD as the LDS of its block tiles allows: three for the 3D FP64
// form, at 137 registers)
template <typename R, int D>
__global__ void __launch_bounds__(kTile, ((D == 3 && sizeof(R) == 8) ? 3 : 1))
k_visc_prep(ViscArgs<R, D> a) {
  extern __shared__ __align__(32) unsigned char smem_raw[];
  __shared__ int halt;
  const bool herr = halted(a.err);
  const TileInfo ti = tile_info(a.tiles, dispatch_tile());
  if (ti.halo0 >= 0) {
    if constexpr (D == 2) visc_prep_block<R>(a, ti, smem_raw, &halt, herr);
    else visc_prep_block3<R>(a, ti, smem_raw, &halt, herr);
    return;
  }
  visc_prep_tile<R, D>(a, ti, smem_raw, &halt, herr);
}

template <typename R, int D>
struct StageArgs {
  const TileInfo *tiles;
  const int4 *tst;           // tile face stencil LL,L,R,RR
  const int8_t *tdir;        // tile face direction
  const int *halo;           // halo lists of the block tiles
  const uint16_t *slots;     // [Nn][2D] tile-local face slot of each cell face
  const uint8_t *flags;      // [Nn]
  const BlkInfo *blk;
  const DevPhys *phys;
  const Flow32 *flow;        // per block (FP32)
  const double *dt;          // [ncases]
  Pack<R, D> Win;            // stencil state this stage reads
  Pack<R, D> Wout;           // stencil state this stage writes (another buffer)
  Pack<double, D> W64;       // FP64 master: the state at the start of the step
                             // until the last stage writes it (mixed mode)
  Pack<R, D> Rv;             // frozen viscous residual
  // SA closure (turb != 0): working variable in the same buffer roles
  const R *nuin;
  R *nuout;
  double *nu64;
  const R *mutf;             // [Nn] frozen face-flux term of the step
  const double *signdis;
  const float *sd32;         // signdis in FP32 (mixed mode)
  int turb;
  MlpDev mlp;                // learned closure (the ML instantiation only)
  unsigned long long *mlcount;   // [2] cells on the network / on the fallback
  double alpha;
  int limiter;
  int last;                  // last stage: residual partials (+ W64 in mixed)
  double *rpart;             // [ntiles][kRpart]
  double *src;               // optional probe [N][5] written at the last stage
  double *nusrc;             // optional probe [N] (SA source, last stage)
  unsigned long long *err;
  // first stage of a step: the frozen viscous residual of the tile first
  // (the work of k_visc_prep, into the same Rv / mutf arrays)
  int fuse_visc;
  ViscArgs<R, D> va;
  // persistent schedule (the P instantiations): gridDim.x workgroups loop
  // over the ntile tiles of the launch (XCD-contiguous runs), with the
  // learned closure's weights staged once per workgroup at byte mlw_off of
  // the dynamic LDS
  int ntile;
  unsigned mlw_off;
  // optional coarse/fine balance (last stage): tile face -> entry of rbal
  // (-1: none); rbal NULL when the balance is off or not this stage's
  const int *tmod;
  const R *rbal;
};

// The fused first stage for the 2D FP64 variant only.  There the viscous
// part needs fewer registers than the stage and the fused launch saves most
// of the separate pass (1.14 -> 1.10 ms per step on the 2.6M-cell NACA0015
// SA case).  In the FP32 variants the separate k_visc_prep runs at a higher
// occupancy than the stage kernel, and fusing measured even (plain closure)
// or slower (learned closure: +100 us on the first stage); in 3D it would
// lower the occupancy of every stage launch.
template <typename R, int D>
constexpr bool kFuseVisc = (D == 2 && std::is_same<R, double>::value);

constexpr int kRpart = 12;   // per tile: max[5], sumsq[5], SA max, SA sumsq
// learned-closure cell counters: kMlSlots pairs (network, fallback), one
// 128-byte line apart, each workgroup adding into slot blockIdx % kMlSlots;
// the reader sums the slots
constexpr int kMlSlots = 64, kMlSlotStride = 16;

// LDS of the learned-closure part of k_stage, after the face fluxes (it
// overwrites the face-cell indices, dead by then; the fluxes are read after
// the network): W1t as 64 rows of its 8 used columns, W2p (64 rows of 64,
// 16-byte chunks XOR-swizzled by the row, see mlp_fwd_reg), b1, b2 and the
// bf16 w3.
constexpr size_t kStageMlSmem = (size_t)64 * 8 * 2 + (size_t)64 * 64 * 2 + 2 * 64 * 4 + 64 * 2;
// byte offset of that region in a block tile: over its states; in 3D the
// cells' residuals follow it
template <int D>
__host__ __device__ constexpr size_t blk_ml_offset() {
  return D == 2 ? blk_state_offset(sizeof(float)) : blk3_state_offset(sizeof(float));
}
template <int D>
__host__ __device__ constexpr size_t blk_ml_smem() {
  return blk_ml_offset<D>() + kStageMlSmem + (D == 3 ? (size_t)kTile * 5 * sizeof(double) : 0);
}
// byte offset of that region for a tile of nface faces (16-byte aligned)
template <typename R, int D>
__host__ __device__ constexpr size_t ml_smem_offset(int nface) {
  return ((sizeof(typename V4<R>::T) + (D == 3 ? sizeof(R) : 0)) * (size_t)nface + 15) & ~(size_t)15;
}

// One workgroup per tile of Morton-consecutive normal cells of one
// (case, level).  Phase 1: every face touching the tile — MUSCL + all-speed
// Roe (NS_Solver.H:704-832) — into LDS (with the SA closure, also the two
// face cells' indices; phase 2 gathers their velocity and working variable
// from cache, phase 1 having just read them).  Phase 2: ComptSource
// (NS_Solver.cpp:282-363), ComptMutSource (:632-840), UpdateConsVars
// (:844-985) and ComptNewPrimVar (:3-194) for the tile's cells.  The ML
// instantiation (mixed mode, launched as k_stage_ml) evaluates the
// point-wise SA term with the network for the cells inside its training
// range, between the two halves of phase 2, on MFMA.  The 2D FP64 first
// stage of a time-march step also does the viscous pass of the tile first
// (fuse_visc).
//
// Win and Wout are different buffers, so no workgroup reads a state another
// one has already advanced within the launch.  U_old is cons(W64): the
// master holds the step-start state until the last stage rewrites it, and
// each cell's master entry is read and written by the same thread.
// The network's weights to LDS at dst (W1t rows' 8 used columns, then W2p
// as stored, b1, b2, the bf16 w3), in 16-byte chunks with all loads issued
// before the stores.  Cooperative over the workgroup; the caller syncs.
__device__ __forceinline__ void ml_fill_weights(const MlpDev &M, unsigned char *dst_raw) {
  __bf16 *mW1t = reinterpret_cast<__bf16 *>(dst_raw);   // [64][8]
  __bf16 *mW2p = mW1t + 64 * 8;                          // [64][64]
  float *mb1 = reinterpret_cast<float *>(mW2p + 64 * 64), *mb2 = mb1 + 64;
  __bf16 *mw3 = reinterpret_cast<__bf16 *>(mb2 + 64);
  constexpr int kW1Rows = 64, kWChunks = kW1Rows + 64 * 64 * 2 / 16;
  static_assert(kWChunks == 576, "weight chunk count");
  uint4 *dst = reinterpret_cast<uint4 *>(mW1t);   // W2p follows W1t in LDS
  const uint4 *s2 = reinterpret_cast<const uint4 *>(M.W2p);   // chunks [64, 576)
  // chunk id of W1t or W2p; both indices stay in range whichever is read
  auto chunk = [&](int id) {
    const uint4 x1 = *reinterpret_cast<const uint4 *>(M.W1t + (size_t)(id < kW1Rows ? id : 0) * kX);
    const uint4 x2 = s2[id < kW1Rows ? 0 : id - kW1Rows];
    return id < kW1Rows ? x1 : x2;
  };
  if (blockDim.x == 256) {
    // chunks t, t+256 always exist; t+512 for t < 64
    const int t = threadIdx.x;
    const uint4 c0 = chunk(t);
    const uint4 c1 = s2[t + 256 - kW1Rows];
    const uint4 c2 = s2[(t < kWChunks - 512 ? t + 512 : 512) - kW1Rows];
    dst[t] = c0;
    dst[t + 256] = c1;
    if (t < kWChunks - 512) dst[t + 512] = c2;
  } else {
    for (int id = threadIdx.x; id < kWChunks; id += blockDim.x) dst[id] = chunk(id);
  }
  for (int i = threadIdx.x; i < 64; i += blockDim.x) {
    mw3[i] = (__bf16)M.w3[i]; mb1[i] = M.b1[i]; mb2[i] = M.b2[i];
  }
}

// Reduction of 16 per-lane slots over a wave: slots 0..7 by maximum, 8..15
// by sum.  A butterfly that halves the slots a lane keeps at each exchange
// (offsets 32, 16, 8, 4: 8 + 4 + 2 + 1 exchanges; the lane with the offset's
// bit set keeps the upper half, so after the first exchange lanes 0..31
// hold maxima and lanes 32..63 sums), then two exchanges of the one slot
// left: lane l returns slot l / 4 of the whole wave.  17 exchanges instead
// of 6 per slot.  The partner of an exchange has the same slot set (their
// lanes differ only in bits not yet used), so each slot combines the same
// 64 values as a per-slot reduction, in another order.
__device__ __forceinline__ double wave_slots16(double *v) {
  const int lane = threadIdx.x & 63;
  const bool sum = (lane & 32) != 0;
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    const double lo = v[j], hi = v[j + 8];
    const double keep = sum ? hi : lo, send = sum ? lo : hi;
    const double o = __shfl_xor(send, 32, 64);
    v[j] = sum ? keep + o : fmax(keep, o);
  }
#pragma unroll
  for (int m = 4, off = 16; m >= 1; m >>= 1, off >>= 1) {
    const bool up = (lane & off) != 0;
#pragma unroll
    for (int j = 0; j < m; ++j) {
      const double lo = v[j], hi = v[j + m];
      const double keep = up ? hi : lo, send = up ? lo : hi;
      const double o = __shfl_xor(send, off, 64);
      v[j] = sum ? keep + o : fmax(keep, o);
    }
  }
  double x = v[0];
#pragma unroll
  for (int off = 2; off >= 1; off >>= 1) {
    const double o = __shfl_xor(x, off, 64);
    x = sum ? x + o : fmax(x, o);
  }
  return x;
}

// Static LDS of a stage workgroup.  halt: the error word is loaded at kernel
// start, its load in flight while the face phase runs, published by thread 0
// just before the face phase's barrier and tested after it (the face phase
// writes only LDS).
struct StageShared {
  int halt;
  unsigned mlc[2];   // learned closure: network / fallback cells of this tile
  double red[kRpart][kTile / 64];
};

// |u|^2 (FP64 mode; fused as written in every variant of the tile)
template <int D>
__device__ __forceinline__ double sq_speed(double u, double v, double w) {
#pragma clang fp contract(off)
  double q = fma(u, u, v * v);
  if (D == 3) q = fma(w, w, q);
  return q;
}

// One tile.  WRES: the network's weights are resident at a.mlw_off
// (persistent schedule); otherwise the ML instantiation stages them after
// the face fluxes, over what is dead by then (a general tile's face-cell
// indices, a block tile's states).  BLK: a block tile (ibg_block.h).
template <typename R, int D, bool ML, bool WRES, bool BLK>
__device__ __forceinline__ void stage_tile(const StageArgs<R, D> &a, const TileInfo &ti, int tile,
                                           bool herr, StageShared &sh) {
  constexpr bool wres = WRES;
  constexpr int NV = D + 2;
  constexpr bool kMixed = std::is_same<R, float>::value;
  using V = typename V4<R>::T;
  extern __shared__ __align__(32) unsigned char smem_raw[];
  int &halt = sh.halt;
  unsigned(&mlc)[2] = sh.mlc;
  auto &red = sh.red;
  if (ML && threadIdx.x == 0) { mlc[0] = 0u; mlc[1] = 0u; }
  auto &bi = uni(a.blk)[ti.blk];
  auto &P = uni(a.phys)[bi.case_id];
  const auto &F32 = uni(a.flow)[ti.blk];
  PhysR<R> ph;
  R ar0, ar1, ar2, ih0, ih1, ih2;
  if constexpr (kMixed) {
    ph = phys_r32(F32);
    ar0 = F32.area[0]; ar1 = F32.area[1]; ar2 = F32.area[2];
    ih0 = F32.invh[0]; ih1 = F32.invh[1]; ih2 = F32.invh[2];
  } else {
    ph = phys_r<R>(P);
    ar0 = bi.area[0]; ar1 = bi.area[1]; ar2 = bi.area[2];
    ih0 = bi.invh[0]; ih1 = bi.invh[1]; ih2 = bi.invh[2];
  }
  V *fl4 = reinterpret_cast<V *>(smem_raw);
  R *fl1 = reinterpret_cast<R *>(smem_raw + sizeof(V) * (size_t)ti.nface);   // 3D 5th value
  // SA: the low / high cell of each face; the cell phase gathers their
  // velocity and working variable (cache hits: phase 1 has just read them)
  int *fL = reinterpret_cast<int *>(smem_raw + (sizeof(V) + (D == 3 ? sizeof(R) : 0)) * (size_t)ti.nface);
  int *fR = fL + ti.nface;
  const BlockLds<R> bl = block_lds<R>(smem_raw, a.turb);
  // this thread's cell in a block tile; after the face phase the ML
  // instantiation forms it anew at each use (held across the network it costs
  // registers that spill)
  const int bp0 = (BLK && D == 2) ? block_cell() : 0;
  auto my_p = [&]() {
    if constexpr (!ML) return bp0;
    int i = threadIdx.x, x, y;
    asm volatile("" : "+v"(i));
    blk_xy(i, x, y);
    return box_pos(x, y);
  };
  const Block3Lds<R> b3 = block3_lds<R>(smem_raw, kBox3Cells);
  // the per-cell arrays from the tile's first cell on, entry c: a uniform base
  // and a 32-bit offset; the flag in flight through the face phase
  const bool live = BLK || (int)threadIdx.x < ti.ncell;
  const int c0 = ti.cell0;
  const unsigned c = live ? threadIdx.x : 0u;
  const uint8_t fg = live ? (a.flags + c0)[c] : 0;
  double s[NV];   // residual of the cell
#pragma unroll
  for (int k = 0; k < NV; ++k) s[k] = 0.0;
  if constexpr (BLK && D == 3) {
    if (threadIdx.x == 0) halt = herr ? 1 : 0;
    block3_load<R, false>(a.Win, a.nuin, a.turb, a.halo, ti, R(0), b3);
    int cx, cy, cz;
    blk_xyz(threadIdx.x, cx, cy, cz);
    __syncthreads();
    // phase 1, one direction at a time: the low face of every cell and the
    // last layer's high faces (each direction's by another wave), then the
    // direction's part of the cells' residuals
    auto direction = [&](auto dc) {
      constexpr int d = decltype(dc)::value;
      block3_faces<d>(cx, cy, cz, [&](int x, int y, int z) {
        int q[4];
        const int p = box3_in(x, y, z);
        if constexpr (d < 2) {
          constexpr int st = d == 0 ? 1 : 12;
          q[0] = p - 2 * st; q[1] = p - st; q[2] = p; q[3] = p + st;
        } else {
          const int hz = box3_zhalo(x, y, 0);   // planes -1, 4, -2, 5 follow, 64 apart
          q[0] = z >= 2 ? p - 2 * kBox3Plane : hz + (z == 1 ? 0 : 128);
          q[1] = z >= 1 ? p - kBox3Plane : hz;
          q[2] = z <= 3 ? p : hz + 64;
          q[3] = z <= 2 ? p + kBox3Plane : hz + (z == 3 ? 64 : 192);
        }
        R flux[5];
        roe_flux<3, d, kMixed>(box3_prim<R>(b3, q[0]), box3_prim<R>(b3, q[1]), box3_prim<R>(b3, q[2]),
                       box3_prim<R>(b3, q[3]), d, d == 0 ? ar0 : (d == 1 ? ar1 : ar2), ph, a.limiter, flux);
        V o;
        o.x = flux[0]; o.y = flux[1]; o.z = flux[2]; o.w = flux[3];
        const int k = flux3_slot(d, x, y, z);
        b3.F.put(k, o);
        b3.Fe[k] = flux[4];
      });
      __syncthreads();
      const int k = flux3_slot(d, cx, cy, cz), h = flux3_slot(d, cx + (d == 0), cy + (d == 1), cz + (d == 2));
      const V lo = b3.F[k], hi = b3.F[h];
      s[0] += (double)lo.x - (double)hi.x;
      s[1] += (double)lo.y - (double)hi.y;
      s[2] += (double)lo.z - (double)hi.z;
      s[3] += (double)lo.w - (double)hi.w;
      s[NV - 1] += (double)b3.Fe[k] - (double)b3.Fe[h];
      sum_now(s);
      if (d < 2) __syncthreads();   // the next direction rewrites the fluxes
    };
    direction(std::integral_constant<int, 0>());
    direction(std::integral_constant<int, 1>());
    direction(std::integral_constant<int, 2>());
  } else if constexpr (BLK) {
    bool loaded = false;
    if constexpr (kFuseVisc<R, D>) {
      if (a.fuse_visc && a.va.viscous) {
        block_load<R, true>(a.Win, a.nuin, a.turb, a.halo, ti, kHalo, (R)P.Rg, bl, bp0);
        __syncthreads();
        block_visc_faces<R>(bl, visc_phys<R, 2>(a.va, ti.blk), a.turb, bp0);
        loaded = true;
      }
      if (a.fuse_visc) {
        // each thread reads back only its own cell's entries in phase 2
        if (threadIdx.x == 0) halt = herr ? 1 : 0;
        __syncthreads();
        if (halt) return;
        block_visc_cell<R>(a.va, ti, bi, P, bl, bp0);
        __syncthreads();   // the face arrays are reused by phase 1
      }
    }
    if (!loaded) {
      block_load<R, false>(a.Win, a.nuin, a.turb, a.halo, ti, kHalo, R(0), bl, bp0);
      __syncthreads();
    }
    // phase 1
    block_faces(bp0, [&](auto dc, int dir, int p) {
      constexpr int d = decltype(dc)::value;
      const int st = dir == 0 ? 1 : kBoxP;
      R flux[4];
      roe_flux<2, d, kMixed>(box_prim<R>(bl, p - 2 * st), box_prim<R>(bl, p - st), box_prim<R>(bl, p),
                             box_prim<R>(bl, p + st), dir, dir == 0 ? ar0 : ar1, ph, a.limiter, flux);
      V o;
      o.x = flux[0]; o.y = flux[1]; o.z = flux[2]; o.w = flux[3];
      bl.fx.put(p - box_pos(0, 0) + (dir == 0 ? 0 : kFxSlots), o);
    });
  } else {
    if constexpr (kFuseVisc<R, D>) {
      if (a.fuse_visc) {
        // Rv and mutf of this tile's cells from the step-start state (the
        // buffer this stage reads); each thread reads back only its own
        // cell's entries in phase 2, so no other workgroup is involved
        visc_prep_tile<R, D>(a.va, ti, smem_raw, &halt, herr);
        if (halt) return;  // uniform: read after the barrier in visc_prep_tile
        __syncthreads();   // the face arrays are reused by phase 1
      }
    }
    for (int f = threadIdx.x; f < ti.nface; f += blockDim.x) {
      const int4 st = a.tst[ti.face0 + f];
      const int dir = a.tdir[ti.face0 + f];
      const Prim<R, D> q0 = pload<R, D>(a.Win, st.x);
      const Prim<R, D> q1 = pload<R, D>(a.Win, st.y);
      const Prim<R, D> q2 = pload<R, D>(a.Win, st.z);
      const Prim<R, D> q3 = pload<R, D>(a.Win, st.w);
      R flux[NV];
      roe_flux<D>(q0, q1, q2, q3, dir, dir == 0 ? ar0 : (dir == 1 ? ar1 : ar2), ph, a.limiter, flux);
      if (a.rbal) {
        // a coarse/fine face of the optional balance: its balanced flux
        const int q = a.tmod[ti.face0 + f];
        if (q >= 0)
          for (int v = 0; v < NV; ++v) flux[v] = a.rbal[(size_t)q * NV + v];
      }
      V o;
      o.x = flux[0]; o.y = flux[1]; o.z = flux[2]; o.w = flux[3];
      fl4[f] = o;
      if (D == 3) fl1[f] = flux[4];
      if (a.turb) {
        fL[f] = st.y;
        fR[f] = st.z;
      }
    }
  }
  if constexpr (!(BLK && D == 3)) {
    if (threadIdx.x == 0) halt = herr ? 1 : 0;
    __syncthreads();
  }
  if (halt) return;   // uniform: the flag was written before the barrier

  const double level_ts = a.alpha * uni(a.dt)[bi.case_id] * bi.step_num;
  // The cell's operands of phase 2, all in flight at once: left at their uses
  // the master would wait for the SA source, and all of them for the flag
  // (the learned closure spills with them held across the network).  The
  // moving FP64 section 72.4 -> 71.1 ms, 3D mixed 52.3 -> 50.4; even where
  // eight waves hide it (2D FP32), and within the 6 % spread of a small mesh's
  // steps.
  constexpr bool kAhead = !ML;
  Prim<double, D> w0;
  R sd_c = R(0), mutf_c = R(0);
  double nu_old = 0.0;
  if constexpr (kAhead) {
    w0 = pload<double, D>(rebase(a.W64, c0), c);
    if (a.turb) {
      sd_c = kMixed ? (R)(a.sd32 + c0)[c] : (R)(a.signdis + c0)[c];
      mutf_c = (a.mutf + c0)[c];
      nu_old = (a.nu64 + c0)[c];
    }
    asm volatile("" ::: "memory");
  }
  // ---- phase 2a: residual of the cell, the SA terms
  double snu = 0.0;
  bool sa_on = false;
  bool use_ml = false;
  R ml_x[kMlpIn];
  R ml_scale = R(0), sa_rest = R(0), sa_nu = R(0);
  // the cell's face slots in the tile's face list
  auto load_slots = [&](int *sl) {
    if (D == 2) {
      const ushort4 s4 = reinterpret_cast<const ushort4 *>(a.slots + (size_t)c0 * 4)[c];
      sl[0] = s4.x; sl[1] = s4.y; sl[2] = s4.z; sl[3] = s4.w;
    } else {
#pragma unroll
      for (int q = 0; q < 2 * D; ++q) sl[q] = (a.slots + (size_t)c0 * 2 * D)[c * 2 * D + q];
    }
  };
  int sl[2 * D];
  if (!BLK && live) load_slots(sl);
  // ComptSource: per direction (F_lo - F_hi), plus the frozen viscous
  // residual sum_d (Fv_hi - Fv_lo).  The learned-closure instantiation
  // forms it after the network (slots read again), so that neither the sum
  // nor the slots are held in registers across the network (they spill).
  auto residual = [&]() {
    if constexpr (ML && !BLK) load_slots(sl);
    int bp = 0;
    if constexpr (BLK && D == 2) bp = my_p() - box_pos(0, 0);
#pragma unroll
    for (int d = 0; d < ((BLK && D == 3) ? 0 : D); ++d) {
      V lo, hi;
      if constexpr (BLK) {
        lo = d == 0 ? bl.fx[bp] : bl.fy[bp];
        hi = d == 0 ? bl.fx[bp + 1] : bl.fy[bp + kBoxP];
      } else {
        lo = fl4[sl[2 * d]];
        hi = fl4[sl[2 * d + 1]];
      }
      s[0] += (double)lo.x - (double)hi.x;
      s[1] += (double)lo.y - (double)hi.y;
      s[2] += (double)lo.z - (double)hi.z;
      s[3] += (double)lo.w - (double)hi.w;
      if (D == 3) s[4] += (double)fl1[sl[2 * d]] - (double)fl1[sl[2 * d + 1]];
    }
    R rv[NV];
    vload<R, D>(rebase(a.Rv, c0), c, rv);
#pragma unroll
    for (int k = 0; k < NV; ++k) s[k] += (double)rv[k];
  };
  if (live) {
    if constexpr (!ML) residual();
    // ComptMutSource for a non-solid updated cell (zero otherwise: the
    // reference never writes mutsource of solid cells)
    if (a.turb && (fg & F_UPDATE) && (fg & F_SA)) {
      sa_on = true;
      Prim<R, D> me;
      int bp = 0, bx = 0, by = 0, bz = 0;
      if constexpr (BLK && D == 2) {
        bp = my_p();
        me = box_prim<R>(bl, bp);
      } else if constexpr (BLK) {
        blk_xyz(threadIdx.x, bx, by, bz);
        me = box3_prim<R>(b3, box3_in(bx, by, bz));
      } else {
        me = pload<R, D>(rebase(a.Win, c0), c);
      }
      R nl[3], nr[3], ul[3], ur[3], vl[3], vr[3], wl[3], wr[3];
#pragma unroll
      for (int d = 0; d < 3; ++d) {
        if (BLK && D == 3) {
          const int p = box3_in(bx, by, bz), hz = box3_zhalo(bx, by, 0);
          const int lp = d == 0 ? p - 1 : (d == 1 ? p - 12 : (bz > 0 ? p - kBox3Plane : hz));
          const int rp = d == 0 ? p + 1 : (d == 1 ? p + 12 : (bz < 3 ? p + kBox3Plane : hz + 64));
          const V lo = b3.S[lp], hi = b3.S[rp];
          ul[d] = lo.y; vl[d] = lo.z; wl[d] = lo.w;
          ur[d] = hi.y; vr[d] = hi.z; wr[d] = hi.w;
          nl[d] = b3.nu[lp];
          nr[d] = b3.nu[rp];
        } else if (BLK && d < D) {
          const int p = bp, st = d == 0 ? 1 : kBoxP;
          const V lo = bl.S[p - st], hi = bl.S[p + st];
          ul[d] = lo.y; vl[d] = lo.z; wl[d] = R(0);
          ur[d] = hi.y; vr[d] = hi.z; wr[d] = R(0);
          nl[d] = bl.nu[p - st];
          nr[d] = bl.nu[p + st];
        } else if (d < D) {
          const int lo = fL[sl[2 * d]], hi = fR[sl[2 * d + 1]];
          uvw_load<R, D>(a.Win, lo, ul[d], vl[d], wl[d]);
          uvw_load<R, D>(a.Win, hi, ur[d], vr[d], wr[d]);
          nl[d] = a.nuin[lo];
          nr[d] = a.nuin[hi];
        } else {
          ul[d] = ur[d] = vl[d] = vr[d] = wl[d] = wr[d] = nl[d] = nr[d] = R(0);
        }
      }
      const R T = v_div(me.p, me.r * ph.Rg);
      const R nu = !BLK ? (a.nuin + c0)[c] : (D == 2 ? bl.nu[bp] : b3.nu[box3_in(bx, by, bz)]);
      const R sd = kAhead ? sd_c : (kMixed ? (R)(a.sd32 + c0)[c] : (R)(a.signdis + c0)[c]);
      const R mutf = kAhead ? mutf_c : (a.mutf + c0)[c];
      SaPhys<R> sp;
      if constexpr (kMixed) sp = sa_phys32(F32);
      else sp = sa_phys(P);
      if constexpr (!ML) {
        snu = (double)sa_source<R, D>(me.u, me.v, me.w, T, me.r, nu, sd, nl, nr, ul, ur, vl, vr,
                                      wl, wr, ih0, ih1, ih2, sp, mutf);
      } else {
        const R h = R(0.5);
        const R i0 = ih0, i1 = ih1, i2 = ih2;
        VelGrad<R> g;
        g.dux = ((ur[0] - ul[0]) * h) * i0; g.dvx = ((vr[0] - vl[0]) * h) * i0; g.dwx = ((wr[0] - wl[0]) * h) * i0;
        g.duy = ((ur[1] - ul[1]) * h) * i1; g.dvy = ((vr[1] - vl[1]) * h) * i1; g.dwy = ((wr[1] - wl[1]) * h) * i1;
        if (D == 3) {
          g.duz = ((ur[2] - ul[2]) * h) * i2; g.dvz = ((vr[2] - vl[2]) * h) * i2; g.dwz = ((wr[2] - wl[2]) * h) * i2;
        } else {
          g.duz = g.dvz = g.dwz = R(0);
        }
        const R dvisx = ((nr[0] - nl[0]) * h) * i0, dvisy = ((nr[1] - nl[1]) * h) * i1;
        const R dvisz = (D == 3) ? ((nr[2] - nl[2]) * h) * i2 : R(0);
        const R olen = sa_olen<R>(g, sp);
        const R mu0 = v_sqrt(T * T * T) * v_div(sp.SoT1, T + sp.SoT);
        // derivative terms in their discrete form
        sa_rest = -(me.u * dvisx + me.v * dvisy + me.w * dvisz) +
                  over_re(v_div(R(SA::cb2) * (dvisx * dvisx + dvisy * dvisy + dvisz * dvisz), R(SA::segma)), sp) +
                  mutf;
        sa_nu = nu;
        bool ok = sa_features<R>(me.u, me.v, me.w, me.r, me.p, mu0, nu, sd, g, olen, sp.Re,
                                 (R)P.init[4], ml_x, ml_scale);
        // the range test without short-circuit branches (a chain of
        // exec-mask branches, one per bound, otherwise)
#pragma unroll
        for (int k = 0; k < kMlpIn; ++k)
          ok = ok & (ml_x[k] >= uni(a.mlp.flo)[k]) & (ml_x[k] <= uni(a.mlp.fhi)[k]);
        use_ml = ok;
        if (!ok) snu = (double)(sa_rest + sa_pointwise<R>(nu, mu0, me.r, sd, olen, sp));
      }
    }
  }
  // ---- learned closure: the network for the cells in its range
  if constexpr (ML) {
    unsigned char *wbase = smem_raw + (wres ? (size_t)a.mlw_off
                                       : BLK ? blk_ml_offset<D>() : ml_smem_offset<R, D>(ti.nface));
    // a 3D block's residual waits in LDS behind the weights (in registers it
    // spills across the network)
    double *keep = reinterpret_cast<double *>(smem_raw + (wres ? (size_t)a.mlw_off : blk_ml_offset<D>()) + kStageMlSmem);
    if (!wres) __syncthreads();   // every phase-2a read of what the weights overwrite is done
    if constexpr (BLK && D == 3) {
#pragma unroll
      for (int k = 0; k < NV; ++k) keep[k * kTile + threadIdx.x] = s[k];
    }
    if (!wres) {
      ml_fill_weights(a.mlp, wbase);
      __syncthreads();
    }
    __bf16 *mW1t = reinterpret_cast<__bf16 *>(wbase);   // [64][8]
    __bf16 *mW2p = mW1t + 64 * 8;                        // [64][64]
    float *mb1 = reinterpret_cast<float *>(mW2p + 64 * 64), *mb2 = mb1 + 64;
    __bf16 *mw3 = reinterpret_cast<__bf16 *>(mb2 + 64);
    const int lane = threadIdx.x & 63;
    bf16x8_t xf;
#pragma unroll
    for (int k = 0; k < kMlpIn; ++k)
      xf[k] = (__bf16)(use_ml ? ((float)ml_x[k] - uni(a.mlp.fmean)[k]) * uni(a.mlp.finv)[k] : 0.0f);
    float yown = 0.0f;
    // one 32-cell block per pass, skipped (wave-uniformly) when none of its
    // cells is on the network; the compiler barrier keeps the weight
    // fragments from being hoisted out of the loop
    const unsigned long long on = __ballot(use_ml);
#pragma unroll 1
    for (int sb = 0; sb < 2; ++sb) {
      asm volatile("" ::: "memory");
      if (((on >> (32 * sb)) & 0xffffffffull) == 0ull) continue;
      const float y = mlp_fwd_reg<8>(xf, sb, mW1t, mW2p, mb1, mb2, mw3);
      if ((lane >> 5) == sb) yown = y;
    }
    if (use_ml) {
      const float z = uni(a.mlp.zst)[0] + uni(a.mlp.zst)[1] * (yown + uni(a.mlp.b3)[0]);
      snu = (double)(sa_rest + (R)z * ml_scale);
    }
    if (a.last && a.mlcount) {
      // cells on the network / on the fallback in this tile (LDS sums,
      // added to the device counters once per workgroup below)
      unsigned long long nm = __ballot(use_ml), nf = __ballot(sa_on && !use_ml);
      if (lane == 0) {
        atomicAdd(&mlc[0], (unsigned)__popcll(nm));
        atomicAdd(&mlc[1], (unsigned)__popcll(nf));
      }
    }
    if constexpr (BLK && D == 3) {
#pragma unroll
      for (int k = 0; k < NV; ++k) s[k] = keep[k * kTile + threadIdx.x];
    }
    if (live) residual();   // (2D and general tiles) the face fluxes are still in LDS
  }
  // ---- phase 2b: update
  if (live) {
    bool write = false;
    double wr = 0, wu = 0, wv = 0, ww = 0, wp = 0;
    double nu_new = 0.0;
    if (fg & F_UPDATE) {
      // U_old = cons(W64): Get_Cons_Vars FlowVariables.H:43-48,
      // e = Cv T + |u|^2/2, T = p/(roe Rg)
      double U[NV];
      {
        if constexpr (!kAhead) w0 = pload<double, D>(rebase(a.W64, c0), c);
        double re0;
        if constexpr (kMixed) {
          const double ke0 = (D == 3) ? 0.5 * (w0.u * w0.u + w0.v * w0.v + w0.w * w0.w)
                                      : 0.5 * (w0.u * w0.u + w0.v * w0.v);
          re0 = w0.r * (P.Cv * n_div(w0.p, w0.r * P.Rg) + ke0);
        } else {
          // roe T = p / Rg
          re0 = fma(P.cvR, w0.p, fma(P.cvRl, w0.p, w0.r * (0.5 * sq_speed<D>(w0.u, w0.v, w0.w))));
        }
        U[0] = w0.r; U[1] = w0.r * w0.u; U[2] = w0.r * w0.v;
        if (D == 3) { U[3] = w0.r * w0.w; U[4] = re0; } else U[3] = re0;
      }
      // cv_old + source * level_ts / v  (NS_Solver.cpp:870)
      const double sc = kMixed ? level_ts * bi.invvol : c_div(level_ts, bi.vol, bi.invvol);
#pragma unroll
      for (int k = 0; k < NV; ++k) U[k] = fma(s[k], sc, U[k]);
      if (a.turb) {
        // viseddy = max(c_vis_old + mutsource * level_ts, 0) (:874-876, :955-957)
        nu_new = (kAhead ? nu_old : (a.nu64 + c0)[c]) + snu * level_ts;
        nu_new = (nu_new < 0.0) ? 0.0 : nu_new;
      }
      if (U[0] < 0.0) report_error(a.err, c0 + (int)c, (fg & F_FINEST) ? 611 : 523);
      if (fg & F_PRIM) {
        // Get_Prim_Vars FlowVariables.H:50-57
        wr = U[0];
        if constexpr (kMixed) {
          const double ir = n_div(1.0, U[0]);
          wu = U[1] * ir;
          wv = U[2] * ir;
          if (D == 3) ww = U[3] * ir;
          const double ke = (D == 3) ? 0.5 * (wu * wu + wv * wv + ww * ww) : 0.5 * (wu * wu + wv * wv);
          wp = (U[D == 3 ? 4 : 3] * ir - ke) * (P.gama - 1.0) * wr;
        } else {
          // the quotients share one reciprocal, each with its exact residual
          // added back
          const double ir = n_rcp(U[0]);
          auto over_r = [&](double x) {
            const double q = x * ir;
            return fma(fma(-U[0], q, x), ir, q);
          };
          wu = over_r(U[1]);
          wv = over_r(U[2]);
          if (D == 3) ww = over_r(U[3]);
          const double ke = 0.5 * sq_speed<D>(wu, wv, ww);
          wp = fma(-ke, wr, U[D == 3 ? 4 : 3]) * (P.gama - 1.0);
        }
        // T = p/(roe Rg) < 0  (NS_Solver.cpp:55-66), Rg > 0
        if ((wp < 0.0) != (wr < 0.0)) report_error(a.err, c0 + (int)c, 37);
        write = true;
      }
    }
    if (!(fg & F_PRIM) && (fg & F_FREE)) {
      // m_data = initvar, the working variable included
      wr = P.init[0]; wu = P.init[1]; wv = P.init[2]; ww = P.init[3]; wp = P.init[4];
      nu_new = P.nut_inf;
      write = true;
    }
    if (write) {
      pstore<R, D>(rebase(a.Wout, c0), c, (R)wr, (R)wu, (R)wv, (R)ww, (R)wp);
      if (kMixed && a.last) pstore<double, D>(rebase(a.W64, c0), c, wr, wu, wv, ww, wp);
    }
    if (a.turb && ((fg & F_UPDATE) || (fg & F_FREE))) {
      (a.nuout + c0)[c] = (R)nu_new;
      if (kMixed && a.last) (a.nu64 + c0)[c] = nu_new;
    }
    if (a.last) {
      if (a.src) {
        double *o = a.src + (size_t)(c0 + (int)c) * 5;
        o[0] = s[0]; o[1] = s[1]; o[2] = s[2];
        if (D == 3) { o[3] = s[3]; o[4] = s[4]; } else { o[3] = 0.0; o[4] = s[3]; }
      }
      if (a.nusrc) (a.nusrc + c0)[c] = snu;
      if (fg & F_RESID) {
        bool nan = (snu != snu);
#pragma unroll
        for (int k = 0; k < NV; ++k) nan = nan || (s[k] != s[k]);
        // a NaN residual aborts the march (ResinDomain, NS_Solver.H:355-375)
        if (nan) report_error(a.err, c0 + (int)c, 268);
      }
    }
  }
  if (a.last) {
    // the wave's partials as 16 slots: maxima (|s_k|, then |snu|) in 0..7,
    // sums of squares in the same order in 8..15, zeros in the rest
    const bool counted = live && (fg & F_RESID);
    double v[16];
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const double x = counted ? (j < NV ? s[j < NV ? j : 0] : (j == NV ? snu : 0.0)) : 0.0;
      v[j] = fabs(x);
      v[8 + j] = x * x;
    }
    const double r = wave_slots16(v);
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
    if ((lane & 3) == 0) {
      // lane 4 s holds slot s of the whole wave
      const int sl = lane >> 2, j = sl & 7;
      if (j < NV) red[sl < 8 ? j : 5 + j][wid] = r;
      else if (j == NV) red[sl < 8 ? 10 : 11][wid] = r;
    }
    __syncthreads();
    // the tile's partials, one entry per thread: entries 0..4 the maxima of
    // (roe, u, v, w, e) (in 2D w is 0 and e the fourth variable), 5..9 the
    // sums of squares, 10 and 11 the working variable's
    if (threadIdx.x < kRpart) {
      const int nw = (blockDim.x + 63) >> 6;
      const int j = threadIdx.x, jv = j < 10 ? j % 5 : 0;
      const int k = (j >= 10) ? j : ((D == 3) ? jv : (jv == 4 ? 3 : (jv == 3 ? -1 : jv)));
      double r = 0.0;
      if (k >= 0) {
        const int row = (j >= 10) ? j : (j < 5 ? k : 5 + k);
        const bool is_max = (j < 5) || (j == 10);
        for (int w = 0; w < nw; ++w) r = is_max ? fmax(r, red[row][w]) : r + red[row][w];
      }
      a.rpart[(size_t)tile * kRpart + j] = r;
    }
    if (threadIdx.x == kRpart) {
      if constexpr (ML) {
        if (a.mlcount) {
          unsigned long long *slot = a.mlcount + (size_t)(blockIdx.x % kMlSlots) * kMlSlotStride;
          if (mlc[0]) atomicAdd(&slot[0], (unsigned long long)mlc[0]);
          if (mlc[1]) atomicAdd(&slot[1], (unsigned long long)mlc[1]);
        }
      }
    }
  }
}

// Schedule P (a separate instantiation each, so that the loop costs the
// one-workgroup-per-tile kernels no registers).  Persistent: XCD x (blocks
// b = x mod 8) owns the x-th contiguous run of the launch's tiles and its
// workgroups take them in turn, so concurrently processed tiles are
// Morton neighbours sharing that XCD's L2.
template <typename R, int D, bool ML, bool P>
__device__ __forceinline__ void stage_launch(const StageArgs<R, D> &a) {
  __shared__ StageShared sh;
  auto one = [&](int tile) {
    const bool herr = halted(a.err);
    const TileInfo ti = tile_info(a.tiles, tile);
    if (ti.halo0 >= 0) {
      stage_tile<R, D, ML, P, true>(a, ti, tile, herr, sh);
      return;
    }
    stage_tile<R, D, ML, P, false>(a, ti, tile, herr, sh);
  };
  if constexpr (!P) {
    one(dispatch_tile());
    return;
  }
  extern __shared__ __align__(32) unsigned char smem_raw[];
  if constexpr (ML) {
    ml_fill_weights(a.mlp, smem_raw + a.mlw_off);
    __syncthreads();
  }
  constexpr int kXcd = 8;
  const int b = (int)blockIdx.x, x = b % kXcd, G = (int)gridDim.x;
  const int per = a.ntile / kXcd, rem = a.ntile % kXcd;
  const int t0 = x * per + (x < rem ? x : rem), t1 = t0 + per + (x < rem ? 1 : 0);
  const int nwk = (G - x + kXcd - 1) / kXcd;   // workgroups of XCD x
  for (int t = t0 + b / kXcd; t < t1; t += nwk) {
    // nothing is hoisted out of the loop: values kept live across the
    // tiles would cost the loop body registers (and occupancy)
    asm volatile("" ::: "memory");
    one(t);
    __syncthreads();   // the next tile rewrites the face arrays
  }
}

// Waves per SIMD the stage kernels are compiled for (the LDS of their block
// tiles allows as many)
template <typename R, int D>
constexpr int kStageWaves = sizeof(R) == 4 ? (D == 2 ? 8 : 6) : (D == 2 ? 4 : 3);

// The persistent variants: what the loop keeps live across its tiles costs
// them registers, and held to more waves they spill and lose (0.9M cells in
// 3D, a march of 32 steps: FP32 9.7 ms at two waves, 7.9 at three, 10.5 at
// five; FP64 18.5 at one, 14.5 at two).
template <typename R, int D>
constexpr int kPersistWaves = sizeof(R) == 4 ? (D == 2 ? 4 : 3) : 2;

template <typename R, int D, bool ML, bool P = false>
__global__ void __launch_bounds__(kTile, (P ? kPersistWaves<R, D> : kStageWaves<R, D>))
k_stage(StageArgs<R, D> a) {
  stage_launch<R, D, ML, P>(a);
}

// The learned-closure stage at seven waves per SIMD: its network needs more
// than the 64 registers eight waves allow (held to 64, the compiler spills
// to scratch and the launch takes 112 instead of 93 us on the 2.6M-cell
// NACA0015 case).
template <int D, bool P = false>
__global__ void __launch_bounds__(kTile) __attribute__((amdgpu_waves_per_eu(P ? 4 : 7, 8)))
k_stage_ml(StageArgs<float, D> a) {
  stage_launch<float, D, true, P>(a);
}

// Stages with a single substep write into buffer 1; this copies the marched
// cells back into the home buffer afterwards.
template <typename R, int D>
__global__ void k_copy_back(int n, Pack<R, D> src, Pack<R, D> dst, const R *nusrc, R *nudst,
                            const unsigned long long *err) {
  const int c = blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= n || halted(err)) return;
  dst.a[c] = src.a[c];
  if (D == 3) dst.e[c] = src.e[c];
  if (nudst) nudst[c] = nusrc[c];
}

// ---------------------------------------------------------- ghost fills
// BCBoxTreat BCValues.H:51-188: -13 pressure inlet (:191-206), -12 pressure
// outlet (:208-214), -50 outflow (:216-220), -81 wall of the TURBULENCE
// build (:89-125); entries (cell, refcell, type, case).  SA working
// variable: copied with the state for -12/-50, the inlet value for -13
// (:203-205), kappa y+ at a wall.
template <int D>
__global__ void k_bc(int n, const int4 *dmg, const DmgWall *wall, StateOut<D> o,
                     const DevPhys *phys) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const bool stop = halted(o.err);   // in flight with the entry
  const int4 e = dmg[i];
  const int g = e.x, ty = e.z;
  const DevPhys &P = phys[e.w];
  const Prim<double, D> q = pload<double, D>(o.m, e.y);
  if (stop) return;
  if (ty == -81) {
    // the wall of the TURBULENCE build (BCValues.H:89-125); nothing in the
    // laminar build, where the branch does not exist
    if (!o.nm || !wall) return;
    const DmgWall W = wall[i];
    if (W.dnbr > 1.0) {
      put_all<D>(o, g, q.r, q.u, q.v, q.w, q.p);
      put_nu<D>(o, g, o.nm[e.y]);
      return;
    }
    // ImageViseddy_Domain Turbulence.cpp:140-195 with the reference cell's
    // neighbour as the reference point and a wall at rest
    const Prim<double, D> s = pload<double, D>(o.m, W.nbr);
    const double *nm = W.nmv;
    const double Tr = s.p / (s.r * P.Rg);
    const double ib_rdis = W.dref / W.dnbr;
    const double hvn = s.u * nm[0] + s.v * nm[1] + s.w * nm[2];
    const double hn[3] = {hvn * nm[0], hvn * nm[1], hvn * nm[2]};
    const double ht[3] = {s.u - hn[0], s.v - hn[1], s.w - hn[2]};
    const double df_velt = sqrt(ht[0] * ht[0] + ht[1] * ht[1] + ht[2] * ht[2]);
    const double hg_mu = sqrt(Tr * Tr * Tr) * ((1.0 + P.SoT) / (Tr + P.SoT));
    const double hg_vis = hg_mu / s.r;
    const double hg_re = df_velt * W.dnbr / hg_vis * P.Re;
    const double hg_yplus = sa_yplus(hg_re);
    const double ut = hg_yplus * hg_vis / W.dnbr / P.Re;
    const double yplus = ib_rdis * hg_yplus;
    const double uplus = sa_uplus(yplus);
    const double ib_velt = uplus * ut;
    const double ib_r0 = (fabs(df_velt) < 0.00000001) ? 0.0 : ib_velt / df_velt;
    double ou[3];
    for (int k = 0; k < 3; ++k) ou[k] = hn[k] * ib_rdis + ht[k] * ib_r0;
    put_all<D>(o, g, s.p / (P.Rg * Tr), ou[0], ou[1], (D == 3) ? ou[2] : 0.0, s.p);
    put_nu<D>(o, g, SA::kappa * yplus);
    return;
  }
  if (ty == -50) {
    put_all<D>(o, g, q.r, q.u, q.v, q.w, q.p);
    if (o.nm) put_nu<D>(o, g, o.nm[e.y]);
  } else if (ty == -12) {
    const double T = q.p / (q.r * P.Rg);
    const double p = P.outlet_p;
    put_all<D>(o, g, p / (P.Rg * T), q.u, q.v, q.w, p);
    if (o.nm) put_nu<D>(o, g, o.nm[e.y]);
  } else if (ty == -13) {
    const double speed0 = sqrt(q.u * q.u + q.v * q.v + q.w * q.w);
    const double u = speed0 * P.inlet_cos, v = speed0 * P.inlet_sin;
    const double T = P.inlet_T0 - (0.5 * (u * u + v * v)) / P.Cp;
    const double p = P.inlet_p0 * pow((T / P.inlet_T0), 3.5);
    put_all<D>(o, g, p / (P.Rg * T), u, v, 0.0, p);
    put_nu<D>(o, g, P.nut_inlet);
  }
}

// The ghost fills below run on a few thousand entries: a chain of memory
// latencies each, so every load that does not depend on another is issued at
// once (the error word with the list entry, the case index with the cell's)
// and the word is tested before the writes.

// PairRestriction[_2d] TwoLevelOp.H:217-231 with AverageCell[_2d] :45-87
// (the SA variant :129-179 averages the working variable without weights).
// cc: (coarse cell, case).
template <int D>
__global__ void k_restrict(int n, const int2 *cc, const int4 *fi, StateOut<D> o, int twod,
                           const DevPhys *phys) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const bool stop = halted(o.err);
  const int2 c = cc[i];
  const int4 f0 = fi[2 * (size_t)i], f1 = fi[2 * (size_t)i + 1];
  const int son[8] = {f0.x, f0.y, f0.z, f0.w, f1.x, f1.y, f1.z, f1.w};
  const DevPhys &P = phys[c.y];
  double r = 0, ru = 0, rv = 0, rw = 0, re = 0, nu = 0;
  auto add = [&](const Prim<double, D> &s, double nv) {
    const double T = s.p / (s.r * P.Rg);
    const double q2 = (D == 3) ? s.u * s.u + s.v * s.v + s.w * s.w : s.u * s.u + s.v * s.v;
    const double e = fma(0.5, q2, P.Cv * T);
    r += s.r;
    ru += s.u * s.r;
    rv += s.v * s.r;
    rw += s.w * s.r;
    re += e * s.r;
    nu += nv;
  };
  // every son's loads in flight, then the sums in son order
  Prim<double, D> s[8];
  double nv[8];
#pragma unroll
  for (int q = 0; q < 8; ++q)
    if (!(twod && (q & 1))) {
      s[q] = pload<double, D>(o.m, son[q]);
      nv[q] = o.nm ? o.nm[son[q]] : 0.0;
    }
#pragma unroll
  for (int q = 0; q < 8; ++q)
    if (!(twod && (q & 1))) add(s[q], nv[q]);
  if (stop) return;
  const double u = ru / r, v = rv / r, w = (D == 3) ? rw / r : 0.0, e = re / r;
  const double rho = r * (twod ? 0.25 : 0.125);
  const double ke = (D == 3) ? 0.5 * (u * u + v * v + w * w) : 0.5 * (u * u + v * v);
  const double p = (e - ke) * (P.gama - 1.0) * rho;
  put_all<D>(o, c.x, rho, u, v, w, p);
  if (o.nm) put_nu<D>(o, c.x, nu * (twod ? 0.25 : 0.125));
}

// PairProlongation[_2d] TwoLevelOp.H:183-215: central gradients of the
// conserved variables over the 6 face neighbours (cneib, :352-358), sons at
// +-1/4 (fincrem); the SA variant (:91-127) does the same for the working
// variable.  One thread per son; cc: (coarse cell, case), nb[6][stride]: the
// cell's neighbours x low, x high, y, z, both listed per pair.  For the 4.4K
// pairs of a level of the moving section 10.5 -> 4.5 us (one thread per
// pair, the neighbours from the cell's row of 27).
template <int D>
__global__ void k_prolong(int n, const int2 *cc, const int *fi, const int *nb, int stride,
                          StateOut<D> o, int twod, const DevPhys *phys) {
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  const int ns = twod ? 4 : 8;
  const int i = t / ns, sn = t - i * ns;
  if (i >= n) return;
  const bool stop = halted(o.err);
  const int2 c = cc[i];
  const int si = twod ? sn >> 1 : sn >> 2, sj = twod ? sn & 1 : (sn >> 1) & 1, sk = twod ? 0 : sn & 1;
  const int f = fi[(size_t)i * 8 + si * 4 + sj * 2 + sk];
  const int ax0 = nb[i], ax1 = nb[stride + i], ay0 = nb[2 * stride + i], ay1 = nb[3 * stride + i];
  const int az0 = twod ? 0 : nb[4 * stride + i], az1 = twod ? 0 : nb[5 * stride + i];
  const DevPhys &P = phys[c.y];
  auto cons = [&](const Prim<double, D> &q, double *U) {
    const double T = q.p / (q.r * P.Rg);
    const double q2 = (D == 3) ? q.u * q.u + q.v * q.v + q.w * q.w : q.u * q.u + q.v * q.v;
    const double e = fma(P.Cv, T, 0.5 * q2);
    U[0] = q.r; U[1] = q.r * q.u; U[2] = q.r * q.v; U[3] = q.r * q.w; U[4] = q.r * e;
  };
  const Prim<double, D> qc = pload<double, D>(o.m, c.x);
  const Prim<double, D> qx0 = pload<double, D>(o.m, ax0), qx1 = pload<double, D>(o.m, ax1);
  const Prim<double, D> qy0 = pload<double, D>(o.m, ay0), qy1 = pload<double, D>(o.m, ay1);
  Prim<double, D> qz0 = qc, qz1 = qc;
  if (!twod) { qz0 = pload<double, D>(o.m, az0); qz1 = pload<double, D>(o.m, az1); }
  double nc = 0, ngx = 0, ngy = 0, ngz = 0;
  if (o.nm) {
    nc = o.nm[c.x];
    ngx = (o.nm[ax1] - o.nm[ax0]) * 0.5;
    ngy = (o.nm[ay1] - o.nm[ay0]) * 0.5;
    if (!twod) ngz = (o.nm[az1] - o.nm[az0]) * 0.5;
  }
  double Uc[5], Ux0[5], Ux1[5], Uy0[5], Uy1[5], Uz0[5], Uz1[5];
  cons(qc, Uc);
  cons(qx0, Ux0); cons(qx1, Ux1);
  cons(qy0, Uy0); cons(qy1, Uy1);
  if (!twod) { cons(qz0, Uz0); cons(qz1, Uz1); }
  const double ix = si ? 0.25 : -0.25, iy = sj ? 0.25 : -0.25, iz = sk ? 0.25 : -0.25;
  double U[5];
  for (int t2 = 0; t2 < 5; ++t2) {
    const double gx = (Ux1[t2] - Ux0[t2]) * 0.5, gy = (Uy1[t2] - Uy0[t2]) * 0.5;
    if (twod) U[t2] = Uc[t2] + ix * gx + iy * gy;
    else U[t2] = Uc[t2] + ix * gx + iy * gy + iz * ((Uz1[t2] - Uz0[t2]) * 0.5);
  }
  if (stop) return;
  const double r = U[0], u = U[1] / r, v = U[2] / r, w = (D == 3) ? U[3] / r : 0.0, e = U[4] / r;
  const double ke = (D == 3) ? 0.5 * (u * u + v * v + w * w) : 0.5 * (u * u + v * v);
  const double p = (e - ke) * (P.gama - 1.0) * r;
  put_all<D>(o, f, r, u, v, w, p);
  if (o.nm) put_nu<D>(o, f, twod ? nc + ix * ngx + iy * ngy : nc + ix * ngx + iy * ngy + iz * ngz);
}

// Body::IBConditions_Image Body.cpp:1366-1496: image state from the
// bracketing cells (Mesh::IntpHGgcellVar Mesh.cpp:1532-1547).  Laminar:
// LinearDist (Body.cpp:183-204) for signdis >= 0, the mirror otherwise.  SA
// closure: ImageViseddy (Turbulence.cpp:57-138, a wall function on the
// tangential velocity, Crocco-Busemann wall temperature, nu = kappa y+) for
// signdis >= 0, and initvar with the wall velocity otherwise
// (Body.cpp:1403-1407).  The image cells of an IB cell are never IB cells
// (checked at upload), so one pass equals the reference's compute-all-then-
// write-all.
template <int D>
__global__ void k_ib(int n, const int *ndev, const int *cell, const int *intp, const double *coef,
                     const double *hgdis, const double *attach, const double *nvec, const int *body,
                     const int *ibcase, const double *signdis, const Motion *mot, int have_motion,
                     StateOut<D> o, const DevPhys *phys, unsigned long long *err) {
  // n: list length, or its capacity when the length lives on the device
  // (moving bodies rebuild the list every step)
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  // the entry (its arrays hold n), the list length and the error word at once
  const int nlist = ndev ? ndev[0] : n;
  const bool stop = halted(err);
  const int4 a0 = *reinterpret_cast<const int4 *>(intp + (size_t)i * 8);
  const int4 a1 = *reinterpret_cast<const int4 *>(intp + (size_t)i * 8 + 4);
  const int cs = ibcase[i], c = cell[i];
  const double hg = hgdis[i];
  double cf[8];
#pragma unroll
  for (int q = 0; q < 8; ++q) cf[q] = coef[(size_t)i * 8 + q];
  if (i >= nlist || stop) return;
  const double sd = signdis[c];
  const DevPhys &P = phys[cs];
  const int at8[8] = {a0.x, a0.y, a0.z, a0.w, a1.x, a1.y, a1.z, a1.w};
  double T = 0, p = 0, u = 0, v = 0, w = 0;
  Prim<double, D> img[8];
#pragma unroll
  for (int q = 0; q < 8; ++q)
    if (at8[q] >= 0) img[q] = pload<double, D>(o.m, at8[q]);
#pragma unroll
  for (int q = 0; q < 8; ++q) {
    if (at8[q] < 0) continue;
    const double cq = cf[q];
    const Prim<double, D> &s = img[q];
    T += cq * (s.p / (s.r * P.Rg));
    p += cq * s.p;
    u += cq * s.u;
    v += cq * s.v;
    w += cq * s.w;
  }
  double pv[3] = {0.0, 0.0, 0.0};
  if (have_motion) {
    const Motion M = mot[body[i]];
    const double *at = attach + (size_t)i * 3;
    const double r1[3] = {at[0] - M.center[0], at[1] - M.center[1], at[2] - M.center[2]};
    pv[0] = M.tra[0] + (M.rot[1] * r1[2] - M.rot[2] * r1[1]);
    pv[1] = M.tra[1] + (M.rot[2] * r1[0] - M.rot[0] * r1[2]);
    pv[2] = M.tra[2] + (M.rot[0] * r1[1] - M.rot[1] * r1[0]);
  }
  if (T < 0.0) report_error(err, c, 1050);
  if (!o.nm) {
    double ou, ov, ow;
    if (sd < 0.0) {
      ou = 2.0 * pv[0] - u; ov = 2.0 * pv[1] - v; ow = 2.0 * pv[2] - w;
    } else {
      const double rt = sd + hg;
      const double r0 = sd / rt;
      ou = pv[0] + (u - pv[0]) * r0;
      ov = pv[1] + (v - pv[1]) * r0;
      ow = pv[2] + (w - pv[2]) * r0;
    }
    put_all<D>(o, c, p / (P.Rg * T), ou, ov, (D == 3) ? ow : 0.0, p);
    return;
  }
  if (sd < 0.0) {
    put_all<D>(o, c, P.init[0], pv[0], pv[1], (D == 3) ? pv[2] : 0.0, P.init[4]);
    put_nu<D>(o, c, P.nut_inf);
    return;
  }
  // ImageViseddy
  const double *nm = nvec + (size_t)i * 3;
  const double rho_hg = p / (P.Rg * T);
  const double rt0 = hg + sd;
  const double ib_rdis = sd / rt0;
  const double hvn = u * nm[0] + v * nm[1] + w * nm[2];
  const double hn[3] = {hvn * nm[0], hvn * nm[1], hvn * nm[2]};
  const double ht[3] = {u - hn[0], v - hn[1], w - hn[2]};
  const double wvn = pv[0] * nm[0] + pv[1] * nm[1] + pv[2] * nm[2];
  const double wn[3] = {nm[0] * wvn, nm[1] * wvn, nm[2] * wvn};
  const double wt[3] = {pv[0] - wn[0], pv[1] - wn[1], pv[2] - wn[2]};
  const double df[3] = {ht[0] - wt[0], ht[1] - wt[1], ht[2] - wt[2]};
  const double df_velt = sqrt(df[0] * df[0] + df[1] * df[1] + df[2] * df[2]);
  const double hg_mu = sqrt(T * T * T) * ((1.0 + P.SoT) / (T + P.SoT));
  const double hg_vis = hg_mu / rho_hg;
  const double hg_re = df_velt * rt0 / hg_vis * P.Re;
  const double hg_yplus = sa_yplus(hg_re);
  const double ut = hg_yplus * hg_vis / rt0 / P.Re;
  const double yplus = ib_rdis * hg_yplus;
  const double uplus = sa_uplus(yplus);
  const double ib_velt = uplus * ut;
  const double ib_r0 = (fabs(df_velt) < 0.00000001) ? 0.0 : ib_velt / df_velt;
  double ou[3];
  for (int k = 0; k < 3; ++k) {
    const double ibn = wn[k] + (hn[k] - wn[k]) * ib_rdis;
    const double ibt = wt[k] + df[k] * ib_r0;
    ou[k] = ibn + ibt;
  }
  const double Tib = T + 0.5 * P.pr_cuberoot / P.Cp * (df_velt * df_velt - ib_velt * ib_velt);
  put_all<D>(o, c, p / (P.Rg * Tib), ou[0], ou[1], (D == 3) ? ou[2] : 0.0, p);
  put_nu<D>(o, c, SA::kappa * yplus);
}

// Comptdt NS_Solver.cpp:229-262 per tile: min over the tile's cells of
// CFL V / sum_d (|u_d| + c) A_d (all three directions, also in 2D).
template <int D>
__global__ void __launch_bounds__(kTile) k_cfl(const TileInfo *tiles, Pack<double, D> W64,
                                               const BlkInfo *blk, const DevPhys *phys,
                                               double *cflpart, unsigned long long *err) {
  __shared__ double red[kTile / 64];
  if (wg_halted(err)) return;
  const TileInfo ti = tiles[blockIdx.x];
  const BlkInfo &bi = blk[ti.blk];
  const DevPhys &P = phys[bi.case_id];
  double d0 = 1.0e300;
  if ((int)threadIdx.x < ti.ncell) {
    const int c = ti.cell0 + threadIdx.x;
    const Prim<double, D> q = pload<double, D>(W64, c);
    const double a = sqrt(P.gama * P.Rg * (q.p / (q.r * P.Rg)));
    const double c0 = (fabs(q.u) + a) * bi.area[0];
    const double c1 = (fabs(q.v) + a) * bi.area[1];
    const double c2 = (fabs(q.w) + a) * bi.area[2];
    d0 = P.cfl * bi.vol / (c0 + c1 + c2);
    if (d0 < 0.0) report_error(err, c, 424);
  }
  for (int off = 32; off > 0; off >>= 1) d0 = fmin(d0, __shfl_xor(d0, off, 64));
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = d0;
  __syncthreads();
  if (threadIdx.x == 0) {
    double m = red[0];
    for (int w = 1; w < (int)((blockDim.x + 63) >> 6); ++w) m = fmin(m, red[w]);
    cflpart[blockIdx.x] = m;
  }
}

// dt = min(CFL_dt, dt*dt_ratio) per case, CFL_dt capped at 10000
// (NS_Solver.cpp:198, 263).  One workgroup per case over the case's tile
// range of each level (ct[case][level] = {first, end}).
__global__ void k_dt_final(int L, const int *ct, const double *cflpart, double *dt,
                           const DevPhys *phys, int ncases, const unsigned long long *err) {
  const int cs = blockIdx.x;
  if (cs >= ncases) return;
  __shared__ double red[4];
  if (wg_halted(err)) return;
  double m = 10000.0;
  for (int l = 0; l < L; ++l) {
    const int a = ct[(cs * L + l) * 2], b = ct[(cs * L + l) * 2 + 1];
    for (int t = a + (int)threadIdx.x; t < b; t += blockDim.x) m = fmin(m, cflpart[t]);
  }
  for (int off = 32; off > 0; off >>= 1) m = fmin(m, __shfl_xor(m, off, 64));
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = m;
  __syncthreads();
  if (threadIdx.x == 0) {
    double v = red[0];
    for (int k = 1; k < (int)((blockDim.x + 63) >> 6); ++k) v = fmin(v, red[k]);
    const double d = dt[cs] * phys[cs].dt_ratio;
    dt[cs] = (v < d) ? v : d;
  }
}

// Stencil copies of the FP64 master after ibg_set_state / ibg_set_nut (one
// upload, the conversions on the device).
template <typename R, int D>
__global__ void k_fill_from_master(int n, Pack<double, D> src, Pack<R, D> dst) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const D4 q = src.a[i];
  typename V4<R>::T o;
  o.x = (R)q.x; o.y = (R)q.y; o.z = (R)q.z; o.w = (R)q.w;
  dst.a[i] = o;
  if (D == 3) dst.e[i] = (R)src.e[i];
}
template <typename R>
__global__ void k_fill_nu_from_master(int n, const double *src, R *dst) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) dst[i] = (R)src[i];
}

// The start of a march: both error words clear, the update counters zero.
__global__ void k_march_begin(unsigned long long *err, unsigned long long *err2,
                              unsigned long long *upd, int n) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (upd && i < n) upd[i] = 0ull;
  if (i == 0) { *err = ~0ull; *err2 = ~0ull; }
}
// Its end: the error word and the sum of the update counters (one wave, 64
// slots of the given stride) into pinned host memory.
__global__ void k_march_end(const unsigned long long *err, const unsigned long long *upd, int stride,
                            unsigned long long *out) {
  unsigned long long s = upd ? upd[(size_t)threadIdx.x * stride] : 0ull;
  for (int off = 32; off > 0; off >>= 1) s += __shfl_xor(s, off, 64);
  if (threadIdx.x == 0) { out[0] = *err; out[1] = s; }
}

__global__ void k_fill_u64(unsigned long long *p, int n, unsigned long long v) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = v;
}

// Body::ComptWallForce Body.cpp:460-555, one workgroup per case, summed in
// a fixed order (deterministic).
template <int D>
__global__ void k_forces(int npatch, const int *pcase, const int *intp, const double *coef,
                         const double *hgdis, const double *nv, const double *pc,
                         const double *area, const double *ccenter, const Motion *mot,
                         int have_motion, Pack<double, D> W64, const DevPhys *phys, int turb,
                         double *out) {
  const int c = blockIdx.x;
  const DevPhys &P = phys[c];
  __shared__ double acc[256][12];
  double s[12];
  for (int k = 0; k < 12; ++k) s[k] = 0.0;
  const double *bc = ccenter + (size_t)c * 3;
  for (int i = threadIdx.x; i < npatch; i += blockDim.x) {
    if (pcase[i] != c) continue;
    double T = 0, p = 0, u = 0, v = 0, w = 0;
    for (int q = 0; q < 8; ++q) {
      const int a = intp[(size_t)i * 8 + q];
      if (a < 0) continue;
      const double cq = coef[(size_t)i * 8 + q];
      const Prim<double, D> sp = pload<double, D>(W64, a);
      T += cq * (sp.p / (sp.r * P.Rg));
      p += cq * sp.p;
      u += cq * sp.u;
      v += cq * sp.v;
      w += cq * sp.w;
    }
    const double *x = pc + (size_t)i * 3;
    const double *n = nv + (size_t)i * 3;
    double pv[3] = {0, 0, 0};
    if (have_motion) {
      const Motion M = mot[c];
      const double r1[3] = {x[0] - M.center[0], x[1] - M.center[1], x[2] - M.center[2]};
      pv[0] = M.tra[0] + (M.rot[1] * r1[2] - M.rot[2] * r1[1]);
      pv[1] = M.tra[1] + (M.rot[2] * r1[0] - M.rot[0] * r1[2]);
      pv[2] = M.tra[2] + (M.rot[0] * r1[1] - M.rot[1] * r1[0]);
    }
    const double A = area[i];
    double df0[3], df1[3];
    if (!turb) {
      const double du[3] = {u - pv[0], v - pv[1], w - pv[2]};
      const double dn = du[0] * n[0] + du[1] * n[1] + du[2] * n[2];
      for (int k = 0; k < 3; ++k) {
        df0[k] = ((du[k] - n[k] * dn) / hgdis[i]) * P.mu * A;
        df1[k] = n[k] * (-p * A);
      }
    } else {
      // Patchut (Turbulence.cpp:197-226): wall-function friction velocity
      // and wall temperature; shear = roe_w ut^2 along the slip direction.
      // FiltSinglePatchPressure (Filt.cpp:44-67) has coefficients b = {1,0..},
      // a = {0..} (Filt.cpp:5-6): the identity, so p is used as is.
      const double roe = p / (P.Rg * T);
      const double hv = u * n[0] + v * n[1] + w * n[2];
      const double pn = pv[0] * n[0] + pv[1] * n[1] + pv[2] * n[2];
      double df[3];
      df[0] = (u - n[0] * hv) - (pv[0] - n[0] * pn);
      df[1] = (v - n[1] * hv) - (pv[1] - n[1] * pn);
      df[2] = (w - n[2] * hv) - (pv[2] - n[2] * pn);
      const double dv = sqrt(df[0] * df[0] + df[1] * df[1] + df[2] * df[2]);
      double vt[3] = {0.0, 0.0, 0.0};
      if (!(dv < 1e-8)) { vt[0] = df[0] / dv; vt[1] = df[1] / dv; vt[2] = df[2] / dv; }
      const double hg_mu = sqrt(T * T * T) * ((1.0 + P.SoT) / (T + P.SoT));
      const double hg_re = roe * dv * hgdis[i] / hg_mu * P.Re;
      const double yplus = sa_yplus(hg_re);
      const double ut = yplus * (hg_mu / roe) / hgdis[i] / P.Re;
      const double wall_T = T + 0.5 * P.pr_cuberoot / P.Cp * (dv * dv);
      const double wall_roe = p / (P.Rg * wall_T);
      const double Cf = wall_roe * (ut * ut);
      for (int k = 0; k < 3; ++k) {
        df0[k] = vt[k] * Cf * A;
        df1[k] = n[k] * (-p * A);
      }
    }
    const double dx[3] = {x[0] - bc[0], x[1] - bc[1], x[2] - bc[2]};
    const double dm0[3] = {dx[1] * df0[2] - dx[2] * df0[1], dx[2] * df0[0] - dx[0] * df0[2], dx[0] * df0[1] - dx[1] * df0[0]};
    const double dm1[3] = {dx[1] * df1[2] - dx[2] * df1[1], dx[2] * df1[0] - dx[0] * df1[2], dx[0] * df1[1] - dx[1] * df1[0]};
    for (int k = 0; k < 3; ++k) { s[k] += df1[k]; s[3 + k] += df0[k]; s[6 + k] += dm1[k]; s[9 + k] += dm0[k]; }
  }
  for (int k = 0; k < 12; ++k) acc[threadIdx.x][k] = s[k];
  __syncthreads();
  // twelve threads, one sum each in thread order (one thread for all of them
  // took 50 us of LDS latency)
  __shared__ double t[12];
  if (threadIdx.x < 12) {
    double x = 0.0;
#pragma unroll 16
    for (int j = 0; j < 256; ++j) x += acc[j][threadIdx.x];
    t[threadIdx.x] = x;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int k = 0; k < 3; ++k) {
      // the SA build scales the wall shear by p_ref*area_ref (Body.cpp:547-553)
      const double sr = turb ? P.p_ref_area : P.shear_ref_area;
      out[c * 6 + k] = t[k] * P.p_ref_area + t[3 + k] * sr;
      out[c * 6 + 3 + k] = t[6 + k] * P.p_ref_area + t[9 + k] * sr;
    }
  }
}

// residual finalize: per case, over the tiles of the last march
// out[case*12 + {0..4}] = L-inf, {5..9} = L2 of the flow residual, {10, 11}
// = L-inf, L2 of the SA residual (res_vis_sum of NS_Solver.H:297, 321).
__global__ void k_resid_final(int ntiles, int L, const int *ct, const double *rpart, double *out,
                              int ncases) {
  // one workgroup per case over its tiles of the last march (tiles < ntiles)
  const int cs = blockIdx.x;
  if (cs >= ncases) return;
  __shared__ double red[kRpart][256];
  double m[6] = {0, 0, 0, 0, 0, 0}, q[6] = {0, 0, 0, 0, 0, 0};
  for (int l = 0; l < L; ++l) {
    const int a = ct[(cs * L + l) * 2], b = min(ct[(cs * L + l) * 2 + 1], ntiles);
    for (int t = a + (int)threadIdx.x; t < b; t += blockDim.x) {
      for (int k = 0; k < 5; ++k) {
        m[k] = fmax(m[k], rpart[(size_t)t * kRpart + k]);
        q[k] += rpart[(size_t)t * kRpart + 5 + k];
      }
      m[5] = fmax(m[5], rpart[(size_t)t * kRpart + 10]);
      q[5] += rpart[(size_t)t * kRpart + 11];
    }
  }
  for (int k = 0; k < 6; ++k) { red[k][threadIdx.x] = m[k]; red[6 + k][threadIdx.x] = q[k]; }
  __syncthreads();
  // twelve threads, one entry each in thread order (one thread for all of
  // them took 25 us of LDS latency)
  const int j = threadIdx.x;
  if (j < kRpart) {
    double x = 0.0;
    const bool sum = j >= 6;
#pragma unroll 16
    for (int w = 0; w < 256; ++w) x = sum ? x + red[j][w] : fmax(x, red[j][w]);
    const int k = sum ? j - 6 : j;
    out[cs * kRpart + (k < 5 ? (sum ? 5 + k : k) : (sum ? 11 : 10))] = sum ? sqrt(x) : x;
  }
}

// parity probes: inviscid / viscous flux of every face, [face][5]
template <typename R, int D>
__global__ void k_face_probe(int nface, const int4 *st, const int8_t *dir, const int16_t *fblk,
                             Pack<R, D> W, const BlkInfo *blk, const DevPhys *phys, int lim,
                             double *out) {
  const int f = blockIdx.x * blockDim.x + threadIdx.x;
  if (f >= nface) return;
  constexpr int NV = D + 2;
  const BlkInfo &bi = blk[fblk[f]];
  const DevPhys &P = phys[bi.case_id];
  const PhysR<R> ph = phys_r<R>(P);
  const int4 s = st[f];
  R flux[NV];
  roe_flux<D>(pload<R, D>(W, s.x), pload<R, D>(W, s.y), pload<R, D>(W, s.z),
              pload<R, D>(W, s.w), dir[f], (R)bi.area[dir[f]], ph, lim, flux);
  double *o = out + (size_t)f * 5;
  if (D == 3) { for (int k = 0; k < 5; ++k) o[k] = flux[k]; }
  else { o[0] = flux[0]; o[1] = flux[1]; o[2] = flux[2]; o[3] = 0.0; o[4] = flux[3]; }
}

template <typename R, int D>
__global__ void k_visc_probe(int nface, const int4 *st, const int4 *vst, const int8_t *dir,
                             const int16_t *fblk, Pack<R, D> W, const BlkInfo *blk,
                             const DevPhys *phys, const Flow32 *flow, const R *nu, double *out,
                             double *mout) {
  const int f = blockIdx.x * blockDim.x + threadIdx.x;
  if (f >= nface) return;
  constexpr int NV = D + 2;
  const ViscPhys<R, D> vp = visc_phys<R, D>(blk, phys, flow, fblk[f]);
  const int4 s = st[f];
  Prim<R, D> t[(D == 3) ? 8 : 4];
  const int4 v0 = vst[(size_t)f * (D - 1)];
  t[0] = pload<R, D>(W, v0.x); t[1] = pload<R, D>(W, v0.y); t[2] = pload<R, D>(W, v0.z); t[3] = pload<R, D>(W, v0.w);
  if (D == 3) {
    const int4 v1 = vst[(size_t)f * (D - 1) + 1];
    t[4 % ((D == 3) ? 8 : 4)] = pload<R, D>(W, v1.x);
    t[5 % ((D == 3) ? 8 : 4)] = pload<R, D>(W, v1.y);
    t[6 % ((D == 3) ? 8 : 4)] = pload<R, D>(W, v1.z);
    t[7 % ((D == 3) ? 8 : 4)] = pload<R, D>(W, v1.w);
  }
  R o5[NV];
  R mf = R(0);
  visc_flux_cells<R, D>(pload<R, D>(W, s.y), pload<R, D>(W, s.z), t, dir[f], vp, o5, nu != nullptr,
                        nu ? nu[s.y] : R(0), nu ? nu[s.z] : R(0), &mf);
  if (mout) mout[f] = mf;
  double *o = out + (size_t)f * 5;
  if (D == 3) { for (int k = 0; k < 5; ++k) o[k] = o5[k]; }
  else { o[0] = o5[0]; o[1] = o5[1]; o[2] = o5[2]; o[3] = 0.0; o[4] = o5[3]; }
}

// plain copy (bandwidth / counter calibration probe)
__global__ void k_copy(const F4 *__restrict__ a, F4 *__restrict__ b, long n) {
  for (long i = blockIdx.x * (long)blockDim.x + threadIdx.x; i < n; i += (long)gridDim.x * blockDim.x)
    b[i] = a[i];
}

}  // namespace ibg
