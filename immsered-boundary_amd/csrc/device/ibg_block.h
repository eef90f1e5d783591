// ibg_block.h — block tiles: 256 Morton-consecutive cells that fill an
// aligned 16 x 16 square (2D) or 8 x 8 x 4 box (3D) of their level.
//
// The faces of such a tile, their stencils and the cells' face slots follow
// from the position in the block, so the tile needs no face list: it reads
// its 256 cells and the indices of its halo cells (132 in 2D: two layers on
// each side, one cell at each corner; 592 in 3D) and works from LDS.  A general tile reads
// 17 B per face (33 B in the viscous pass, ~2.2 faces per cell), 8 B of
// slots per cell, and gathers each state record about nine times from
// L1/L2; a block tile reads 2 B per cell of halo indices and each record
// once.  90 % of the cells of the 2.6M-cell section and 80 % of a
// 4.2M-cell ensemble lie in block tiles; the rest, the ragged rims of the
// refinement levels, stay in general tiles (as does a block whose stencils
// are not the regular ones, and every tile of another size than 256 cells).
//
// Average launch, general tiles only -> with block tiles.  2D, moving
// 2.6M-cell section: k_stage FP64 150 -> 134 us, FP32 71 -> 61 us (the
// learned closure's 97 -> 87 us), k_visc_prep FP32 66 -> 43 us (30 with the
// layout below).  3D, 2.7M
// cells: k_stage FP32 147 -> 124 us, FP64 300 -> 294 us, k_visc_prep FP32
// 172 -> 72 us, FP64 321 -> 128 us.  The FP32 stages then issue vector
// instructions for 77 % (3D) to 92 % (2D) of their time (2D: the bytes alone
// would take 36 us at the copy rate), the FP64 ones for 65 to 79 %.  So the
// code spends them sparingly: the limiters without branches, one
// position per thread for every phase, the last column's and row's faces in
// one pass (2D), FP32 constants from a table (Flow32), uniform bases with 32-bit
// offsets.  With those and leaner FP64 arithmetic the 2D stages take 53 us
// (FP32), 81 (learned closure) and 104 (FP64), the 3D ones 111 and 210.
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

// coordinates of halo entry h (-2 .. 17)
__host__ __device__ inline void halo_xy(int h, int &x, int &y) {
  if (h >= kHaloL1 && h < kHaloC) {
    const int c = h - kHaloL1;
    x = (c & 1) ? kBlkN : -1;
    y = (c & 2) ? kBlkN : -1;
    return;
  }
  const int far = h >= kHaloC ? 1 : 0;
  const int k = far ? h - kHaloC : h;
  const int t = k & (kBlkN - 1), side = k >> 4;
  const int o = (side & 1) ? kBlkN + far : -1 - far;
  x = (side & 2) ? t : o;
  y = (side & 2) ? o : t;
}
// box position of halo entry h
__host__ __device__ inline int halo_pos(int h) {
  int x, y;
  halo_xy(h, x, y);
  return box_pos(x, y);
}

// The FP32 viscous pass keeps the square and one halo layer as pairs (u, v),
// (roe, p) and (1 / (roe Rg), working variable): a face reads the velocities
// of six cells and the rest of two, mostly as two neighbouring records by one
// instruction for 16 lanes at a time; at pitch 20 their five rows (or five
// columns) of four 8-byte records lie on distinct banks.  From the stage's
// 16-byte records the reads of (u, v) alone used half the banks: 325 of the
// pass's 585 cycles per wave and CU were bank conflicts, 136 of 450 now; with
// pitch 24 (32 lanes of one record each on distinct banks) 207 of 500.
// 43 -> 30 us on the moving section.
constexpr int kViscP = 20, kViscCells = (kBlkN + 2) * kViscP;
__host__ __device__ constexpr int visc_pos(int x, int y) { return (y + 1) * kViscP + x + 1; }
__host__ __device__ constexpr size_t blk_visc_smem32() {
  return 16 * (size_t)kFluxSlots + 3 * 8 * (size_t)kViscCells;
}

// LDS bytes of a block tile: fluxes, the box's states, with the SA closure
// its working variable, and with `temp` (viscous pass) its temperature
__host__ __device__ constexpr size_t blk_state_offset(size_t rsize) { return 4 * rsize * kFluxSlots; }
__host__ __device__ constexpr size_t blk_smem(size_t rsize, bool turb, bool temp) {
  return blk_state_offset(rsize) + (4 * rsize + (turb ? rsize : 0) + (temp ? rsize : 0)) * kBoxCells;
}

// ------------------------------------------------------------------- 3D
// 8 x 8 x 4 cells (x, y, z), Morton order x lowest.  LDS records of the stage
// kernel: the four planes as 12 x 12 boxes (x and y halos in place), then
// the halo planes z = -1, 4, -2, 5 of 8 x 8 cells; the working variable stops
// before the last two.  The viscous pass keeps the 10 x 10 x 6 box of the
// first halo layer.  The face fluxes of one direction at a time: with all
// three the LDS would hold two workgroups less per CU.
//
// Pitches and slots by the bank rule of 16-byte reads, as measured: the LDS
// serves 16 lanes at a time, lanes 0-3, 12-15, 20-23 and 24-27, then the other
// half of the 32; they must differ in the record's address modulo 16 (x bit 0,
// y bit 0 and pairs of z bit 0, x bit 1, y bit 1 of the Morton order).  Both
// boxes and the three flux layouts satisfy it: 5 cycles per read of 64 lanes;
// 8 and 12 with the box pitches 12 / 152 and 10 / 100 and fluxes at 9 / 76.
// FP64 records are two planes of 16-byte halves.  k_visc_prep FP64 179 -> 148
// us, k_stage FP64 236 -> 229 (2D FP64, for the halves alone, 111 -> 106); in
// FP32 the reads were not what bounds.
constexpr int kB3X = 8, kB3Y = 8, kB3Z = 4;
constexpr int kBox3Plane = 144, kBox3Halo = 4 * kBox3Plane;
constexpr int kBox3Cells = kBox3Halo + 4 * 64, kBox3Nu = kBox3Halo + 2 * 64;
constexpr int kVBox3P = 12, kVBox3Plane = 128, kVBox3Cells = 6 * kVBox3Plane;
constexpr int kFlux3 = 320;
// halo list: layer 1 (x, y, z; low then high side), the edges of the first
// layer (xy, xz, yz; low/low, high/low, low/high, high/high), layer 2
constexpr int kHalo3L1 = 256, kHalo3E = kHalo3L1 + 80, kHalo3 = kHalo3E + 256;

__host__ __device__ inline void blk_xyz(int i, int &x, int &y, int &z) {
  x = (i & 1) | ((i >> 2) & 2) | ((i >> 4) & 4);
  y = ((i >> 1) & 1) | ((i >> 3) & 2) | ((i >> 5) & 4);
  z = ((i >> 2) & 1) | ((i >> 4) & 2);
}
// coordinates of halo entry h (-2 .. 9, -2 .. 9, -2 .. 5)
__host__ __device__ inline void halo3_xyz(int h, int &x, int &y, int &z) {
  if (h >= kHalo3L1 && h < kHalo3E) {
    int k = h - kHalo3L1;
    if (k < 16) {
      z = k & 3; x = (k & 4) ? kB3X : -1; y = (k & 8) ? kB3Y : -1;
    } else if (k < 48) {
      k -= 16;
      y = k & 7; x = (k & 8) ? kB3X : -1; z = (k & 16) ? kB3Z : -1;
    } else {
      k -= 48;
      x = k & 7; y = (k & 8) ? kB3Y : -1; z = (k & 16) ? kB3Z : -1;
    }
    return;
  }
  const int far = h >= kHalo3E ? 1 : 0, k = far ? h - kHalo3E : h;
  const int a = k & 7, b = (k >> 3) & 3, side = (k >> 5) & 1;
  if (k < 64) {
    x = side ? kB3X + far : -1 - far; y = a; z = b;
  } else if (k < 128) {
    y = side ? kB3Y + far : -1 - far; x = a; z = b;
  } else {
    x = a; y = (k >> 3) & 7; z = (k & 64) ? kB3Z + far : -1 - far;
  }
}
__host__ __device__ inline int box3_in(int x, int y, int z) { return z * kBox3Plane + (y + 2) * 12 + x + 2; }
// plane n of the halo planes z = -1, 4, -2, 5
__host__ __device__ inline int box3_zhalo(int x, int y, int n) { return kBox3Halo + n * 64 + y * 8 + x; }
__host__ __device__ inline int box3_pos(int x, int y, int z) {
  if (z >= 0 && z < kB3Z) return box3_in(x, y, z);
  return box3_zhalo(x, y, z == -1 ? 0 : (z == kB3Z ? 1 : (z < 0 ? 2 : 3)));
}
__host__ __device__ constexpr int vbox3_pos(int x, int y, int z) {
  return (z + 1) * kVBox3Plane + (y + 1) * kVBox3P + x + 1;
}
// flux slot of the low face of cell (x, y, z) in direction d
__host__ __device__ constexpr int flux3_slot(int d, int x, int y, int z) {
  return d == 0 ? 32 * x + ((y + 8 * z) ^ ((x & 1) << 2))
                : (d == 1 ? x + 8 * y + 76 * z : 64 * z + ((x + 8 * y) ^ ((z & 1) << 2)));
}

__host__ __device__ constexpr size_t blk3_state_offset(size_t rsize) { return 5 * rsize * kFlux3; }
__host__ __device__ constexpr size_t blk3_smem(size_t rsize, bool turb) {
  return blk3_state_offset(rsize) + 5 * rsize * kBox3Cells + (turb ? rsize * kBox3Nu : 0);
}
__host__ __device__ constexpr size_t blk3_visc_smem(size_t rsize, bool turb) {
  return blk3_state_offset(rsize) + (5 * rsize + (turb ? rsize : 0)) * kVBox3Cells;
}

}  // namespace ibg
