// ibg_block.h — block tiles: 256 Morton-consecutive cells that fill an
// aligned 16 x 16 square of their level (2D).
//
// The faces of such a tile, their stencils and the cells' face slots follow
// from the position in the square, so the tile needs no face list: it reads
// its 256 cells and the indices of its 132 halo cells (two layers on each
// side, one cell at each corner) and works from LDS.  A general tile reads
// 17 B per face (33 B in the viscous pass, ~2.2 faces per cell), 8 B of
// slots per cell, and gathers each state record about nine times from
// L1/L2; a block tile reads 2 B per cell of halo indices and each record
// once.  90 % of the cells of the 2.6M-cell section and 80 % of a
// 4.2M-cell ensemble lie in block tiles; the rest, the ragged rims of the
// refinement levels, stay in general tiles (a level's square that lacks a
// cell, or whose stencil is not the regular one, is general; so are all
// tiles of other sizes than 256 cells and of 3D meshes).  Average launch of
// the moving 2.6M-cell section, general tiles only -> with block tiles:
// k_stage FP64 150 -> 134 us, FP32 71 -> 61 us (the learned closure's 97 ->
// 87 us), k_visc_prep FP32 66 -> 43 us.  The FP32 stage then issues vector
// instructions for about two thirds of its time (its bytes alone would take
// 36 us at the copy rate); the FP64 one for most of it.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace ibg {

constexpr int kBlkN = 16;          // cells per side
constexpr int kBlkCells = 256;
// LDS box of the square and its two halo layers, pitch 20: the 4 x 4 cells
// that 16 consecutive lanes hold (Morton order) start at x + 20 y, that is
// 4 (x + 20 y) dwords for 16-byte records, 16 distinct groups of 4 of the 64
// banks, for any shift of the square
constexpr int kBoxP = 20;
constexpr int kBoxCells = kBoxP * kBoxP;
// face fluxes: 16 rows of 17 x faces (pitch 20), then 17 rows of 16 y faces
constexpr int kFxSlots = kBlkN * kBoxP;
constexpr int kFluxSlots = kFxSlots + (kBlkN + 1) * kBoxP;
// halo list: layer 1 by side (x low, x high, y low, y high), the corners
// (low/low, high/low, low/high, high/high in x/y), layer 2 by side
constexpr int kHaloL1 = 4 * kBlkN, kHaloC = kHaloL1 + 4, kHalo = kHaloC + 4 * kBlkN;

__host__ __device__ constexpr int box_pos(int x, int y) { return (y + 2) * kBoxP + x + 2; }

// square coordinates of cell i (Morton order, x the low bit)
__host__ __device__ inline void blk_xy(int i, int &x, int &y) {
  x = (i & 1) | ((i >> 1) & 2) | ((i >> 2) & 4) | ((i >> 3) & 8);
  y = ((i >> 1) & 1) | ((i >> 2) & 2) | ((i >> 3) & 4) | ((i >> 4) & 8);
}

// box position of halo entry h
__host__ __device__ inline int halo_pos(int h) {
  if (h >= kHaloL1 && h < kHaloC) {
    const int c = h - kHaloL1;
    return box_pos((c & 1) ? kBlkN : -1, (c & 2) ? kBlkN : -1);
  }
  const int far = h >= kHaloC ? 1 : 0;
  const int k = far ? h - kHaloC : h;
  const int t = k & (kBlkN - 1), side = k >> 4;
  const int o = (side & 1) ? kBlkN + far : -1 - far;
  return (side & 2) ? box_pos(t, o) : box_pos(o, t);
}

// LDS bytes of a block tile: fluxes, the box's states, with the SA closure
// its working variable, and with `temp` (viscous pass) its temperature
__host__ __device__ constexpr size_t blk_state_offset(size_t rsize) { return 4 * rsize * kFluxSlots; }
__host__ __device__ constexpr size_t blk_smem(size_t rsize, bool turb, bool temp) {
  return blk_state_offset(rsize) + (4 * rsize + (turb ? rsize : 0) + (temp ? rsize : 0)) * kBoxCells;
}

}  // namespace ibg
