// ibg_closure.h — training-data sampler, training and stand-alone inference
// kernels of the learned SA closure (network in ibg_mlp.h).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "ibg_kernels.h"

namespace ibg {

__device__ __forceinline__ uint64_t mix64(uint64_t x) {
  // splitmix64 finaliser
  x += 0x9e3779b97f4a7c15ull;
  x = (x ^ (x >> 30)) * 0xbf58476d1ce4e5b9ull;
  x = (x ^ (x >> 27)) * 0x94d049bb133111ebull;
  return x ^ (x >> 31);
}

// Central-difference velocity gradient and |Omega| of cell c from the
// Box::neib neighbours (ComptMutSource NS_Solver.cpp:662-703), FP64.
template <int D>
__device__ __forceinline__ VelGrad<double> cell_grad(const Pack<double, D> &W, const int *nb27,
                                                     int c, const BlkInfo &bi) {
  const int *nb = nb27 + (size_t)c * 27;
  const Prim<double, D> xl = pload<double, D>(W, nb[0 * 9 + 1 * 3 + 1]);
  const Prim<double, D> xr = pload<double, D>(W, nb[2 * 9 + 1 * 3 + 1]);
  const Prim<double, D> yl = pload<double, D>(W, nb[1 * 9 + 0 * 3 + 1]);
  const Prim<double, D> yr = pload<double, D>(W, nb[1 * 9 + 2 * 3 + 1]);
  VelGrad<double> g;
  g.dux = (xr.u - xl.u) * 0.5 * bi.invh[0];
  g.dvx = (xr.v - xl.v) * 0.5 * bi.invh[0];
  g.dwx = (xr.w - xl.w) * 0.5 * bi.invh[0];
  g.duy = (yr.u - yl.u) * 0.5 * bi.invh[1];
  g.dvy = (yr.v - yl.v) * 0.5 * bi.invh[1];
  g.dwy = (yr.w - yl.w) * 0.5 * bi.invh[1];
  g.duz = g.dvz = g.dwz = 0.0;
  if (D == 3) {
    const Prim<double, D> zl = pload<double, D>(W, nb[1 * 9 + 1 * 3 + 0]);
    const Prim<double, D> zr = pload<double, D>(W, nb[1 * 9 + 1 * 3 + 2]);
    g.duz = (zr.u - zl.u) * 0.5 * bi.invh[2];
    g.dvz = (zr.v - zl.v) * 0.5 * bi.invh[2];
    g.dwz = (zr.w - zl.w) * 0.5 * bi.invh[2];
  }
  return g;
}

// Training data from the solver's own state: every normal fluid cell that
// the update advances (F_UPDATE, signdis > 0) is kept with probability frac
// (seeded hash of the cell), with its raw features and the target
// z = Q / (nu S^) of the plain closure in FP64.  One workgroup per tile, in
// two passes so that the rows land in a fixed order (tile, then cell):
// kWrite = false stores the tile's count of kept cells, k_closure_offsets
// turns the counts into row offsets after the rows already stored, and
// kWrite = true writes each kept cell at its offset plus its rank in the
// tile.  Rows past the capacity are dropped.
template <int D, bool kWrite>
__global__ void __launch_bounds__(kTile) k_closure_sample(const TileInfo *tiles, const BlkInfo *blk,
                                                         const DevPhys *phys, const uint8_t *flags,
                                                         Pack<double, D> W, const double *nu,
                                                         const double *signdis, const int *nb27,
                                                         double frac, uint64_t seed, float *X,
                                                         float *Z, int *Cell, int *tcount,
                                                         const long long *toff, long long cap) {
  __shared__ int wsum[kTile / 64];
  const TileInfo ti = tiles[blockIdx.x];
  const int c = ti.cell0 + threadIdx.x;
  bool keep = (int)threadIdx.x < ti.ncell && (flags[c] & F_UPDATE) && signdis[c] > 0.0;
  if (keep) {
    const double u01 = (double)(mix64(seed ^ ((uint64_t)c * 0x632be59bd9b4e019ull)) >> 11) *
                       (1.0 / 9007199254740992.0);
    keep = u01 < frac;
  }
  double x[kMlpIn], z = 0.0;
  if (keep) {
    const BlkInfo &bi = blk[ti.blk];
    const DevPhys &P = phys[bi.case_id];
    const Prim<double, D> me = pload<double, D>(W, c);
    const double T = me.p / (me.r * P.Rg);
    const double mu0 = sqrt(T * T * T) * ((1.0 + P.SoT) / (T + P.SoT));
    const VelGrad<double> g = cell_grad<D>(W, nb27, c, bi);
    const double olen = sa_olen<double>(g, sa_phys(P));
    double scale;
    keep = sa_features<double>(me.u, me.v, me.w, me.r, me.p, mu0, nu[c], signdis[c], g, olen,
                               P.Re, P.init[4], x, scale);
    if (keep) z = sa_pointwise<double>(nu[c], mu0, me.r, signdis[c], olen, sa_phys(P)) / scale;
  }
  // rank of the kept cell within the tile: wave prefix + earlier waves
  const unsigned long long bal = __ballot(keep);
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  const int below = __popcll(bal & ((1ull << lane) - 1ull));
  if (lane == 0) wsum[wid] = __popcll(bal);
  __syncthreads();
  int before = 0, total = 0;
  for (int w = 0; w < (int)((blockDim.x + 63) >> 6); ++w) {
    if (w < wid) before += wsum[w];
    total += wsum[w];
  }
  if constexpr (!kWrite) {
    if (threadIdx.x == 0) tcount[blockIdx.x] = total;
  } else {
    if (keep) {
      const long long k = toff[blockIdx.x] + before + below;
      if (k < cap) {
        for (int j = 0; j < kMlpIn; ++j) X[(size_t)k * kMlpIn + j] = (float)x[j];
        Z[k] = (float)z;
        Cell[k] = c;
      }
    }
  }
}

// Exclusive prefix sum of the per-tile counts after the count of rows
// already stored (count[0]), then count[0] += the total.  One workgroup.
__global__ void __launch_bounds__(1024) k_closure_offsets(const int *tcount, int ntiles,
                                                          long long *toff,
                                                          unsigned long long *count) {
  __shared__ long long part[1024];
  const int t = threadIdx.x, nt = blockDim.x;
  const int per = (ntiles + nt - 1) / nt, a = t * per, b = min(ntiles, a + per);
  long long s = 0;
  for (int i = a; i < b; ++i) s += tcount[i];
  part[t] = s;
  __syncthreads();
  if (t == 0) {
    long long run = (long long)count[0];
    for (int k = 0; k < nt; ++k) { const long long v = part[k]; part[k] = run; run += v; }
    count[1] = (unsigned long long)run;   // new total, published below
  }
  __syncthreads();
  long long run = part[t];
  for (int i = a; i < b; ++i) { toff[i] = run; run += tcount[i]; }
  __syncthreads();
  if (t == 0) count[0] = count[1];
}

// Per-block partial moments of the dataset: for each of the 8 features and
// the target: sum, sum of squares, min, max (double).
__global__ void k_closure_moments(const float *X, const float *Z, long long n, double *part) {
  __shared__ double red[256][4];
  double acc[kMlpIn + 1][4];
  for (int j = 0; j <= kMlpIn; ++j) { acc[j][0] = 0; acc[j][1] = 0; acc[j][2] = 1e300; acc[j][3] = -1e300; }
  for (long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x; i < n; i += (long long)gridDim.x * blockDim.x) {
    for (int j = 0; j <= kMlpIn; ++j) {
      const double v = (j < kMlpIn) ? (double)X[i * kMlpIn + j] : (double)Z[i];
      acc[j][0] += v; acc[j][1] += v * v;
      acc[j][2] = fmin(acc[j][2], v); acc[j][3] = fmax(acc[j][3], v);
    }
  }
  for (int j = 0; j <= kMlpIn; ++j) {
    red[threadIdx.x][0] = acc[j][0]; red[threadIdx.x][1] = acc[j][1];
    red[threadIdx.x][2] = acc[j][2]; red[threadIdx.x][3] = acc[j][3];
    __syncthreads();
    if (threadIdx.x == 0) {
      double s = 0, s2 = 0, mn = 1e300, mx = -1e300;
      for (int t = 0; t < (int)blockDim.x; ++t) {
        s += red[t][0]; s2 += red[t][1]; mn = fmin(mn, red[t][2]); mx = fmax(mx, red[t][3]);
      }
      double *o = part + ((size_t)blockIdx.x * (kMlpIn + 1) + j) * 4;
      o[0] = s; o[1] = s2; o[2] = mn; o[3] = mx;
    }
    __syncthreads();
  }
}

// fp32 master parameters -> the bf16 layouts of the kernels.
__global__ void k_closure_pack(const float *p, __bf16 *W1t, __bf16 *W2t, __bf16 *W2, __bf16 *W2p,
                               float *w3, float *b1, float *b2, float *b3) {
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t < 64 * kX) {
    const int j = t / kX, k = t % kX;
    W1t[t] = (__bf16)(k < kMlpIn ? p[kOffW1 + k * 64 + j] : 0.0f);
  }
  if (t < 64 * kH) {
    const int a = t / kH, b = t % kH;
    W2t[t] = (__bf16)(b < 64 ? p[kOffW2 + b * 64 + a] : 0.0f);   // W2t[j][i] = W2[i][j]
    W2[t] = (__bf16)(b < 64 ? p[kOffW2 + a * 64 + b] : 0.0f);    // W2[i][j]
  }
  if (t < 64 * 64) {
    // W2p row j, physical 16-byte chunk pc holds logical chunk pc ^ (j % 8);
    // logical column 16 kt + 8 h + e = W2[pi(kt, h, e)][j] with
    // pi(kt, h, e) = 32 (kt/2) + 8 (2 (kt%2) + e/4) + 4 h + e%4 (mlp_fwd_reg)
    const int j = t / 64, pc = (t % 64) / 8, e = t % 8;
    const int lc = pc ^ (j & 7), kt = lc / 2, hh = lc % 2;
    const int pk = 32 * (kt / 2) + 8 * (2 * (kt % 2) + e / 4) + 4 * hh + e % 4;
    W2p[t] = (__bf16)p[kOffW2 + pk * 64 + j];
  }
  if (t < 64) {
    w3[t] = (float)(__bf16)p[kOffW3 + t];
    b1[t] = p[kOffB1 + t];
    b2[t] = p[kOffB2 + t];
  }
  if (t == 0) b3[0] = p[kOffB3];
}

// Stand-alone inference over raw feature rows: z = zmean + zstd * y, with
// the register forward of the stage kernel (mlp_fwd_reg): 64 rows per wave,
// one row per lane.  X and Z may be pinned host memory: a row is two 16-byte
// loads and a wave's 64 results one 256-byte store, so the rows cross the
// link as the kernel runs (16384 rows in 13.6 us, 43 GB/s: the link bounds
// it).  The weights go to LDS in 16-byte chunks.
__global__ void __launch_bounds__(256) k_closure_infer(MlpDev M, const float *X, float *Zout, long long n) {
  __shared__ __align__(16) unsigned char smem[kStageMlSmem];
  const long long row = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  float x[kMlpIn] = {};
  if (row < n) {
    const float4 x0 = *reinterpret_cast<const float4 *>(X + row * kMlpIn);
    const float4 x1 = *reinterpret_cast<const float4 *>(X + row * kMlpIn + 4);
    x[0] = x0.x; x[1] = x0.y; x[2] = x0.z; x[3] = x0.w;
    x[4] = x1.x; x[5] = x1.y; x[6] = x1.z; x[7] = x1.w;
  }
  ml_fill_weights(M, smem);
  __syncthreads();
  const __bf16 *sW1t = reinterpret_cast<const __bf16 *>(smem), *sW2p = sW1t + 64 * 8;
  const float *sb1 = reinterpret_cast<const float *>(sW2p + 64 * 64), *sb2 = sb1 + 64;
  const __bf16 *sw3 = reinterpret_cast<const __bf16 *>(sb2 + 64);
  bf16x8_t xf;
#pragma unroll
  for (int k = 0; k < kMlpIn; ++k)
    xf[k] = (__bf16)(row < n ? (x[k] - uni(M.fmean)[k]) * uni(M.finv)[k] : 0.0f);
  const int lane = threadIdx.x & 63;
  float yown = 0.0f;
#pragma unroll 1
  for (int sb = 0; sb < 2; ++sb) {
    const float y = mlp_fwd_reg<8>(xf, sb, sW1t, sW2p, sb1, sb2, sw3);
    if ((lane >> 5) == sb) yown = y;
  }
  if (row < n) Zout[row] = uni(M.zst)[0] + uni(M.zst)[1] * (yown + uni(M.b3)[0]);
}

// Forward + backward of 64 rows per workgroup (4 waves x 16 rows), loss
// L = (1/B) sum (y - t)^2 on the standardised target.  Rows come from the
// dataset through a seeded hash (sampling with replacement) or, when
// explicit is set, rows blockIdx.x*64 .. +63 in order (the gradient check).
// Each workgroup writes its full gradient into grad[blockIdx.x][kNParam]
// and its loss sum into lossp[blockIdx.x].
//
// A batch is at most a few hundred workgroups, so a step is one dependent
// chain per wave.  A wave keeps its 16 rows in registers from the gather to
// dZ1: weights come from L2 straight into fragments (issued together with
// the row gather, no staging in LDS), the ReLU derivatives stay where the
// MFMA left them, and each activation is stored transposed as well, four
// rows of a column at a time, so that the weight gradients, which contract
// over rows, read their fragments as 16-byte rows.  One barrier: the
// contractions over all 64 rows.  8192 rows: 16.7 -> 7.9 us (weights and
// row-major activations staged in LDS, fragments gathered 2 bytes at a time,
// nine barriers).  With the Adam kernel below a step takes 52 -> 15 us.
struct TrainArgs {
  MlpDev M;
  const float *X, *Z;
  long long n;         // dataset rows
  int batch;           // B (loss normalisation)
  int explicit_rows;
  uint64_t seed;
  float *grad, *lossp;
};

__global__ void __launch_bounds__(256) k_closure_train(TrainArgs a) {
  typedef __bf16 bf16x4_t __attribute__((ext_vector_type(4)));
  // [row][unit] and, T, [unit][row], both of stride kH
  __shared__ __align__(16) __bf16 sH1[64 * kH], sH1T[64 * kH], sD2[64 * kH], sD2T[64 * kH],
      sH2T[64 * kH], sD1T[64 * kH], sXT[kMlpIn * kH];
  __shared__ __align__(16) float sdy[64], se2[64], part[3][4][64];
  const MlpDev &M = a.M;
  const int w = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int r = lane & 15, q = lane >> 4;
  // this lane's row (its features in the lanes q == 0) and target
  const long long slot = (long long)blockIdx.x * 64 + 16 * w + r;
  const long long row = a.explicit_rows ? slot : (long long)(mix64(a.seed + (uint64_t)slot) % (uint64_t)a.n);
  const bool have = row < a.n;
  // weight fragments
  bf16x8_t w1[4], w2t[2][4], w2[2][4];
  float b1v[4], b2v[4], w3v[4];
#pragma unroll
  for (int nt = 0; nt < 4; ++nt) {
    const int col = 16 * nt + r;
    w1[nt] = *reinterpret_cast<const bf16x8_t *>(M.W1t + col * kX + 8 * q);
    b1v[nt] = M.b1[col]; b2v[nt] = M.b2[col]; w3v[nt] = M.w3[col];
#pragma unroll
    for (int kt = 0; kt < 2; ++kt) {
      w2t[kt][nt] = *reinterpret_cast<const bf16x8_t *>(M.W2t + col * kH + 32 * kt + 8 * q);
      w2[kt][nt] = *reinterpret_cast<const bf16x8_t *>(M.W2 + col * kH + 32 * kt + 8 * q);
    }
  }
  float t = 0.0f;
  bf16x8_t xf = {};
  if (have) {
    t = (a.Z[row] - M.zst[0]) / M.zst[1];
    if (q == 0) {
      const float4 x0 = *reinterpret_cast<const float4 *>(a.X + row * kMlpIn);
      const float4 x1 = *reinterpret_cast<const float4 *>(a.X + row * kMlpIn + 4);
      const float x[kMlpIn] = {x0.x, x0.y, x0.z, x0.w, x1.x, x1.y, x1.z, x1.w};
#pragma unroll
      for (int k = 0; k < kMlpIn; ++k) xf[k] = (__bf16)((x[k] - M.fmean[k]) * M.finv[k]);
    }
  }
  if (q == 0)
#pragma unroll
    for (int k = 0; k < kMlpIn; ++k) sXT[k * kH + 16 * w + r] = xf[k];
  // layer 1
  floatx4_t acc[4];
  unsigned on1 = 0, on2 = 0;   // relu' of the lane's 16 units, bit 4 nt + v
#pragma unroll
  for (int nt = 0; nt < 4; ++nt) {
    acc[nt] = mfma16(xf, w1[nt], floatx4_t{b1v[nt], b1v[nt], b1v[nt], b1v[nt]});
    bf16x4_t h;
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      h[v] = (__bf16)mlp_act(acc[nt][v]);
      on1 |= (acc[nt][v] > 0.0f ? 1u : 0u) << (4 * nt + v);
      sH1[(16 * w + 4 * q + v) * kH + 16 * nt + r] = h[v];
    }
    *reinterpret_cast<bf16x4_t *>(sH1T + (16 * nt + r) * kH + 16 * w + 4 * q) = h;
  }
  __builtin_amdgcn_wave_barrier();   // a wave reads back its own rows: LDS is in order
  // layer 2
#pragma unroll
  for (int nt = 0; nt < 4; ++nt) acc[nt] = floatx4_t{b2v[nt], b2v[nt], b2v[nt], b2v[nt]};
#pragma unroll
  for (int kt = 0; kt < 2; ++kt) {
    const bf16x8_t av = *reinterpret_cast<const bf16x8_t *>(sH1 + (16 * w + r) * kH + 32 * kt + 8 * q);
#pragma unroll
    for (int nt = 0; nt < 4; ++nt) acc[nt] = mfma16(av, w2t[kt][nt], acc[nt]);
  }
  float yv[4] = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
  for (int nt = 0; nt < 4; ++nt) {
    bf16x4_t h;
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      h[v] = (__bf16)mlp_act(acc[nt][v]);
      on2 |= (acc[nt][v] > 0.0f ? 1u : 0u) << (4 * nt + v);
      yv[v] += (float)h[v] * w3v[nt];
    }
    *reinterpret_cast<bf16x4_t *>(sH2T + (16 * nt + r) * kH + 16 * w + 4 * q) = h;
  }
  // y of rows 4 q + v (the same in the 16 lanes of a group), its error and
  // dy = dL/dy; rows past n in the explicit mode contribute nothing
  const float invB = 1.0f / (float)a.batch;
  float dy[4];
#pragma unroll
  for (int v = 0; v < 4; ++v) {
    for (int off = 1; off < 16; off <<= 1) yv[v] += __shfl_xor(yv[v], off, 64);
    const float tv = __shfl(t, 4 * q + v, 64);
    const bool valid = !a.explicit_rows || (long long)blockIdx.x * 64 + 16 * w + 4 * q + v < a.n;
    const float e = valid ? (yv[v] + M.b3[0]) - tv : 0.0f;
    dy[v] = 2.0f * e * invB;
    if (r == 0) {
      sdy[16 * w + 4 * q + v] = dy[v];
      se2[16 * w + 4 * q + v] = e * e;
    }
  }
  // dZ2 = bf16(dy w3 relu'(Z2))
#pragma unroll
  for (int nt = 0; nt < 4; ++nt) {
    bf16x4_t d;
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      d[v] = (__bf16)(dy[v] * w3v[nt] * (float)((on2 >> (4 * nt + v)) & 1u));
      sD2[(16 * w + 4 * q + v) * kH + 16 * nt + r] = d[v];
    }
    *reinterpret_cast<bf16x4_t *>(sD2T + (16 * nt + r) * kH + 16 * w + 4 * q) = d;
  }
  __builtin_amdgcn_wave_barrier();
  // dZ1 = bf16((dZ2 W2^T) relu'(Z1)) for this wave's rows
#pragma unroll
  for (int nt = 0; nt < 4; ++nt) acc[nt] = floatx4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int kt = 0; kt < 2; ++kt) {
    const bf16x8_t av = *reinterpret_cast<const bf16x8_t *>(sD2 + (16 * w + r) * kH + 32 * kt + 8 * q);
#pragma unroll
    for (int nt = 0; nt < 4; ++nt) acc[nt] = mfma16(av, w2[kt][nt], acc[nt]);
  }
#pragma unroll
  for (int nt = 0; nt < 4; ++nt) {
    bf16x4_t d;
#pragma unroll
    for (int v = 0; v < 4; ++v) d[v] = (__bf16)(acc[nt][v] * (float)((on1 >> (4 * nt + v)) & 1u));
    *reinterpret_cast<bf16x4_t *>(sD1T + (16 * nt + r) * kH + 16 * w + 4 * q) = d;
  }
  __builtin_amdgcn_wave_barrier();
  // column sums over the wave's 16 rows, lane = unit: dw3 = sum H2 dy,
  // db2 = sum dZ2, db1 = sum dZ1
  {
    auto rows16 = [&](const __bf16 *T, int half) {
      return *reinterpret_cast<const bf16x8_t *>(T + lane * kH + 16 * w + 8 * half);
    };
    float s3 = 0.0f, s2 = 0.0f, s1 = 0.0f;
#pragma unroll
    for (int half = 0; half < 2; ++half) {
      const bf16x8_t h2 = rows16(sH2T, half), d2 = rows16(sD2T, half), d1 = rows16(sD1T, half);
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        s3 += (float)h2[e] * sdy[16 * w + 8 * half + e];
        s2 += (float)d2[e];
        s1 += (float)d1[e];
      }
    }
    part[0][w][lane] = s3; part[1][w][lane] = s2; part[2][w][lane] = s1;
  }
  __syncthreads();
  float *g = a.grad + (size_t)blockIdx.x * kNParam;
  if (w < 3) {
    g[(w == 0 ? kOffW3 : (w == 1 ? kOffB2 : kOffB1)) + lane] =
        part[w][0][lane] + part[w][1][lane] + part[w][2][lane] + part[w][3][lane];
  } else if (lane < 2) {
    // the loss (lane 0) and db3 = sum dy (lane 1), in row order
    const float4 *p = reinterpret_cast<const float4 *>(lane == 0 ? se2 : sdy);
    float s = 0.0f;
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const float4 v = p[i];
      s += v.x; s += v.y; s += v.z; s += v.w;
    }
    if (lane == 0) a.lossp[blockIdx.x] = s;
    else g[kOffB3] = s;
  }
  // dW2[i][j] = sum_r H1[r][i] dZ2[r][j] and dW1[k][i] = sum_r X[r][k]
  // dZ1[r][i]: wave w -> i in 16w..16w+15
  floatx4_t d1 = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int nt = 0; nt < 4; ++nt) acc[nt] = floatx4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int kt = 0; kt < 2; ++kt) {
    const bf16x8_t zero = {};
    const bf16x8_t av = *reinterpret_cast<const bf16x8_t *>(sH1T + (16 * w + r) * kH + 32 * kt + 8 * q);
#pragma unroll
    for (int nt = 0; nt < 4; ++nt)
      acc[nt] = mfma16(av, *reinterpret_cast<const bf16x8_t *>(sD2T + (16 * nt + r) * kH + 32 * kt + 8 * q), acc[nt]);
    const bf16x8_t xv = *reinterpret_cast<const bf16x8_t *>(sXT + (r & 7) * kH + 32 * kt + 8 * q);
    d1 = mfma16(r < kMlpIn ? xv : zero,
                *reinterpret_cast<const bf16x8_t *>(sD1T + (16 * w + r) * kH + 32 * kt + 8 * q), d1);
  }
#pragma unroll
  for (int nt = 0; nt < 4; ++nt)
#pragma unroll
    for (int v = 0; v < 4; ++v) g[kOffW2 + (16 * w + 4 * q + v) * 64 + 16 * nt + r] = acc[nt][v];
  if (q < 2)
#pragma unroll
    for (int v = 0; v < 4; ++v) g[kOffW1 + (4 * q + v) * 64 + 16 * w + r] = d1[v];
}

// One parameter's entries in the layouts of k_closure_pack.
__device__ __forceinline__ void pack_param(int i, float p, __bf16 *W1t, __bf16 *W2t, __bf16 *W2,
                                           __bf16 *W2p, float *w3, float *b1, float *b2, float *b3) {
  if (i < kOffB1) W1t[(i % 64) * kX + i / 64] = (__bf16)p;
  else if (i < kOffW2) b1[i - kOffB1] = p;
  else if (i < kOffB2) {
    const int in = (i - kOffW2) / 64, j = (i - kOffW2) % 64;
    const __bf16 h = (__bf16)p;
    W2[in * kH + j] = h;
    W2t[j * kH + in] = h;
    // the chunk and element of W2p whose pi(kt, h, e) is `in`
    const int m = in & 31, lc = 2 * (2 * (in >> 5) + ((m >> 4) & 1)) + ((m >> 2) & 1);
    W2p[j * 64 + 8 * (lc ^ (j & 7)) + 4 * ((m >> 3) & 1) + (m & 3)] = h;
  } else if (i < kOffW3) b2[i - kOffB2] = p;
  else if (i < kOffB3) w3[i - kOffW3] = (float)(__bf16)p;
  else b3[0] = p;
}

// Adam over the summed workgroup gradients (beta1 0.9, beta2 0.999, eps
// 1e-8), then the parameter's entries of the kernels' layouts (no separate
// pack launch).  With gsum_out set, only the summed gradient is written.
// The sum runs over the workgroups in order; its loads are independent, 32
// in flight at a time (one at a time, 128 workgroups of gradients took 128
// memory latencies: 31.4 + 4.8 us of repacking -> 6.0 us for 8192 rows), and 64-thread groups
// spread the 4801 parameters over 76 CUs.
constexpr int kAdamThreads = 64;
__global__ void __launch_bounds__(kAdamThreads) k_closure_adam(float *p, float *m, float *v,
                                                               const float *grad, int nwg, float lr,
                                                               int step, float *gsum_out,
                                                               __bf16 *W1t, __bf16 *W2t, __bf16 *W2,
                                                               __bf16 *W2p, float *w3, float *bb1,
                                                               float *bb2, float *bb3) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= kNParam) return;
  constexpr int kFly = 32;
  float g = 0.0f;
  int k = 0;
  for (; k + kFly <= nwg; k += kFly) {
    float x[kFly];
#pragma unroll
    for (int j = 0; j < kFly; ++j) x[j] = grad[(size_t)(k + j) * kNParam + i];
#pragma unroll
    for (int j = 0; j < kFly; ++j) g += x[j];
  }
  if (k < nwg) {
    // the rest, clamped loads so that they too are in flight together
    float x[kFly];
#pragma unroll
    for (int j = 0; j < kFly; ++j) x[j] = grad[(size_t)min(k + j, nwg - 1) * kNParam + i];
#pragma unroll
    for (int j = 0; j < kFly; ++j)
      if (k + j < nwg) g += x[j];
  }
  if (gsum_out) {
    gsum_out[i] = g;
    return;
  }
  const float b1 = 0.9f, b2 = 0.999f;
  const float mi = b1 * m[i] + (1.0f - b1) * g;
  const float vi = b2 * v[i] + (1.0f - b2) * g * g;
  m[i] = mi;
  v[i] = vi;
  const float mh = mi / (1.0f - powf(b1, (float)step));
  const float vh = vi / (1.0f - powf(b2, (float)step));
  const float pn = p[i] - lr * mh / (sqrtf(vh) + 1e-8f);
  p[i] = pn;
  pack_param(i, pn, W1t, W2t, W2, W2p, w3, bb1, bb2, bb3);
}

}  // namespace ibg
