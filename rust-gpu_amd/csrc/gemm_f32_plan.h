// gemm_f32_plan.h — which tile of gemm_f32.h a call runs, and whether the one-launch kernel or the
// conversion passes plus the bf16 GEMM take it; and the kernel's global index maps.  Plain
// arithmetic (no HIP), also compiled into the CPU test of both (tests/gemm_f32_plan_sim.cpp).
#pragma once
#if defined(__HIPCC__)
#include <hip/hip_runtime.h>
#endif
#include <stdint.h>

#include "index_maps.h"

namespace t0mi {

// The products of the Ignis matmul: which operands are K-major (rows of the f32 matrix are K).
enum F32Mode : int {
  F32_FORWARD = 0,  // Y[m,n] = X[m,k] . W[k,n]: right operand K-major
  F32_DATA = 1,     // dX[m,k] = dY[m,n] . W[k,n]^T: neither
  F32_WEIGHT = 2,   // dW[k,n] = X[m,k]^T . dY[m,n]: both
};
inline bool f32_a_kmajor(int mode) { return mode == F32_WEIGHT; }
inline bool f32_b_kmajor(int mode) { return mode != F32_DATA; }

constexpr int kF32Bk = 32;  // K of a tile
// A 128 x 128 tile's second set of sums (gemm_f32.h, fold) would take the registers of the CU's
// second workgroup; it runs only with K per piece up to this.
constexpr bool gemm_f32_folds(int bm, int bn) { return bm * bn < 128 * 128; }
constexpr uint32_t kF32ChainMax = 1024;
constexpr uint32_t kF32MaxPieceWgs = 768;      // workgroups of a launch that cuts K
constexpr uint64_t kF32SlotBytes = 32u << 20;  // exchange slots of such a launch, at most
constexpr uint64_t kF32MaxBytes = 1ull << 31;  // operand extent (32-bit byte offsets)

// The prebuilt tiles and the coefficients of their time (microseconds) on MI355X:
//   t = c[0] + c[1] it + c[2] it (w - 1) + c[3] (w - 1)          it: K tiles per wave group, a tile
//     + [pieces > 1] (c[4] + c[5] wgs / 256 * bm bn / 1024)         whose rows are not whole 128-byte
//     + c[6] MB_out / 8 + c[7] MB_in / 8                             lines counted up to 1.5 times;
//                                                                    w: workgroups on the busiest CU
// Fitted to 864 random calls (m 4..2048, n and k 64..8192, all three products) timed with every
// tile and 1 to 8 pieces; on 857 others the tile picked is 3 % behind the fastest (geometric mean).
struct F32Tiles {
  int bm, bn, groups;
  float c[8];
};
constexpr F32Tiles kF32Tiles[] = {
    {32, 32, 8, {4.268f, 0.632f, 0.871f, 2.287f, 1.208f, 1.554f, 4.706f, 0.577f}},
    {64, 32, 4, {4.057f, 0.468f, 0.658f, 2.130f, 1.284f, 0.848f, 2.525f, 0.308f}},
    {64, 64, 2, {3.907f, 0.316f, 0.396f, 0.804f, 1.763f, 0.224f, 1.574f, 0.509f}},
    {128, 64, 1, {4.087f, 0.261f, 0.280f, 1.031f, 2.295f, 0.218f, 1.020f, 0.376f}},
    {128, 128, 1, {4.767f, 0.285f, 0.460f, 0.795f, 3.346f, 0.235f, 1.118f, 0.697f}},
};
constexpr int kF32TileCount = sizeof kF32Tiles / sizeof kF32Tiles[0];

// The same for a bf16 right operand (Y = X . WT^T, the inference layer on its cached weight), fitted
// to 120 random calls of 1 to 64 rows (n 256..14336, k 256..8192); on 120 others the tile picked is 1 %
// behind the fastest of eight.
constexpr F32Tiles kWtTiles[] = {
    {32, 64, 4, {3.827f, 0.268f, 0.311f, 0.646f, 1.522f, 0.378f, 5.687f, 0.451f}},
    {64, 64, 2, {4.112f, 0.216f, 0.112f, 1.584f, 1.886f, 0.221f, 0.000f, 0.521f}},
};
constexpr int kWtTileCount = sizeof kWtTiles / sizeof kWtTiles[0];
constexpr uint32_t kWtMaxRows = 64;

// First row (column) of the tile that starts at `start`, of `size`, in a matrix of `extent`: a tile
// that would end past the matrix starts earlier.
T0MI_HD constexpr int f32_tile_first(int start, int extent, int size) {
  const int last = extent - size;
  return start < last ? start : last > 0 ? last : 0;
}
// Byte offset at K = 0 of 16-byte piece `sp` of source row r of the tile starting at `first`: K-major
// source rows are K (and the piece 4 columns of the product), others the tile's own rows.  Rows past
// the matrix are past every operand's extent: the range check answers them with zeros and no fetch.
constexpr uint32_t kF32Oob = 0x80000000u;
T0MI_HD constexpr uint32_t f32_piece_off(bool kmajor, uint32_t ld, int first, int rows, int r, int sp) {
  if (kmajor) return ((uint32_t)r * ld + (uint32_t)(first + sp * 4)) * 4u;
  return first + r < rows ? ((uint32_t)(first + r) * ld + (uint32_t)(sp * 4)) * 4u : kF32Oob;
}
// Workgroup `b` of a launch that cuts K over `pieces` workgroups a tile: the tile (its slots, and the order
// in which neighbours share an XCD), the K piece and the number whose counter the tile's pieces share.  False:
// the numbering's padding.  The numbers go past the tiles where these are no multiple of the XCDs; the
// slots do not.
T0MI_HD bool f32_workgroup(uint32_t b, uint32_t nx, uint32_t pieces, uint32_t tiles, uint32_t* tile,
                           uint32_t* piece, uint32_t* counter) {
  xk_unpack(b, nx, pieces, counter, piece);
  *tile = *counter % nx * ((tiles + nx - 1) / nx) + *counter / nx;
  return *tile < tiles;
}
// First K tile of piece q of p over nkt K tiles (piece q ends where q + 1 starts).
T0MI_HD constexpr int f32_piece_begin(int q, int p, int nkt) { return (int)((int64_t)q * nkt / p); }

struct F32Plan {
  int tile = -1;        // index into kF32Tiles; -1: the conversion passes and the bf16 GEMM
  uint32_t pieces = 1;  // workgroups over K per tile
  uint32_t tiles_m = 0, tiles_n = 0;
};

// The conversion passes, the bf16 GEMM with its split-K reduce, and the unpad pass (same data).
inline float f32_two_pass_us(uint32_t m, uint32_t n, uint32_t k) {
  const float mk = (float)m * k, kn = (float)k * n, mn = (float)m * n;
  float t = 10.06f + 1.84f * (mk + kn) * 6e-6f / 8 + 1.236e-9f * 2 * mn * k + 1.56f * mn * 4e-6f / 8;
  if (n % 8) t += 3.5f + 1.75f * mn * 8e-6f / 8;
  return t;
}

// The fastest tile of `tab` (and K pieces; `split`: the in-launch exchange is available) for Y[m,n] over
// K = k, right operand elements of `b_size` bytes, and its time in *us.  A K-major operand narrower
// than the tile needs a multiple of 4 columns (a 16-byte load may then not straddle the matrix's
// end); other operands take any size.
inline F32Plan f32_best_tile(const F32Tiles* tab, int count, int mode, int b_size, uint32_t m, uint32_t n, uint32_t k,
                             uint32_t cus, bool split, float* best_us) {
  F32Plan best;
  if (!m || !n || !k) return best;
  if ((uint64_t)m * k * 4 >= kF32MaxBytes || (uint64_t)k * n * b_size >= kF32MaxBytes) return best;
  if ((uint64_t)m * n * 4 >= 64 * kF32MaxBytes) return best;
  const uint32_t nkt = (k + kF32Bk - 1) / kF32Bk;
  for (int i = 0; i < count; ++i) {
    const F32Tiles& t = tab[i];
    if (f32_a_kmajor(mode) && (int64_t)m < t.bm && m % 4) continue;
    if (f32_b_kmajor(mode) && (int64_t)n < t.bn && n % 4) continue;
    const uint64_t tm = (m + t.bm - 1) / t.bm, tn = (n + t.bn - 1) / t.bn, tiles = tm * tn;
    if (tiles > 65536) continue;  // far past the range where one launch is the faster route
    for (uint32_t p = 1; p <= (split ? 8u : 1u); p *= 2) {
      const uint32_t kt = (nkt + p - 1) / p;  // K tiles of the longest piece
      if (p > 1 && (tiles * p > kF32MaxPieceWgs || tiles * p * t.bm * t.bn * 4 > kF32SlotBytes ||
                    nkt < p * (uint32_t)t.groups))
        break;
      if (!gemm_f32_folds(t.bm, t.bn) && kt * kF32Bk > kF32ChainMax) continue;
      const uint64_t wgs = tiles * p;
      float w = (float)wgs / cus;
      w = w <= 3 ? (float)((wgs + cus - 1) / cus) : w + 0.5f;
      float it = (float)((kt + t.groups - 1) / t.groups);
      if (k % 32)  // K-contiguous rows that start inside a 128-byte line
        it *= 1 + 0.5f * ((f32_a_kmajor(mode) ? 0 : t.bm) + (f32_b_kmajor(mode) ? 0 : t.bn)) / (t.bm + t.bn);
      float us = t.c[0] + t.c[1] * it + (t.c[2] * it + t.c[3]) * (w - 1) + t.c[6] * ((float)m * n) * 4e-6f / 8 +
                 t.c[7] * ((float)m * k * 4 + (float)k * n * b_size) * 1e-6f / 8;
      if (p > 1) us += t.c[4] + t.c[5] * (float)wgs / 256 * (t.bm * t.bn) / 1024;
      if (best.tile < 0 || us < *best_us) {
        best.tile = i;
        best.pieces = p;
        best.tiles_m = (uint32_t)tm;
        best.tiles_n = (uint32_t)tn;
        *best_us = us;
      }
    }
  }
  return best;
}
// The estimates are 10 % off at small sizes and optimistic at large ones, where the routes meet (f32
// weights: about 30 GFLOP): there the one launch has to be that much ahead.
inline bool f32_one_launch_ahead(float us, float other_us) {
  return us + 0.2f * (us > 15 ? us - 15 : 0) <= other_us;
}

// What the estimate leaves out with K in 8 pieces over four and more rows of 128-row tiles: about what was
// measured over what was estimated, some 130 calls with K of 2000 .. 8192.  Held against the passes only where
// these need no padding (their estimate is 4 % high there, and 15 % low with padding).  On 153 other calls
// that it moves to the passes, these are 1.10 times as fast (geometric mean; 8 of them slower by more than
// 2 %, 7 % at most; 696 x 192 x 8128, data: 32.4 -> 21.5 us).  With two or three rows of tiles the same
// correction moved as many calls wrongly as rightly.
inline float f32_wide_pieces(const F32Plan& p, uint32_t n, uint32_t k) {
  if (p.pieces < 8 || kF32Tiles[p.tile].bm < 128 || n % 8 || k % 8 || p.tiles_m < 4) return 1.0f;
  return p.tiles_m >= 5 && p.tiles_m <= 8 ? 1.4f : 1.2f;
}

// Y[m,n] over K = k with f32 operands: a tile of kF32Tiles, or -1.
inline F32Plan f32_plan(int mode, uint32_t m, uint32_t n, uint32_t k, uint32_t cus, bool split) {
  float us = 0;
  F32Plan p = f32_best_tile(kF32Tiles, kF32TileCount, mode, 4, m, n, k, cus, split, &us);
  if (p.tile >= 0) us *= f32_wide_pieces(p, n, k);
  if (p.tile >= 0 && !f32_one_launch_ahead(us, f32_two_pass_us(m, n, k))) p.tile = -1;
  return p;
}

// Y[m,n] = X[m,k] . WT[n,k]^T, X f32, WT bf16 (k % 8 == 0): a tile of kWtTiles, or -1 for X's
// conversion and the bf16 routes.  Their times: up to 16 rows and one round of 16-column units the
// persistent decode kernel (ahead at 1 x 4096 x 4096 alone of what was measured: 9.8 against 10.7
// us), else the scheduled GEMM with its split-K reduce.
inline F32Plan wt_plan(uint32_t m, uint32_t n, uint32_t k, uint32_t cus, bool split) {
  F32Plan p;
  if (m > kWtMaxRows || k % 8) return p;
  float us = 0;
  p = f32_best_tile(kWtTiles, kWtTileCount, F32_DATA, 2, m, n, k, cus, split, &us);
  const bool decode = m <= 16 && k % 32 == 0 && (uint64_t)n <= 16ull * cus;
  const float other = decode ? 6.6f + (float)k * (0.00078f + 0.00005f * (float)(m - 1))
                             : 7.579f + 1.276f * ((float)k * n) * 2e-6f / 8 + 20.56f * ((float)m * k) * 6e-6f / 8;
  if (p.tile >= 0 && !f32_one_launch_ahead(us, other)) p.tile = -1;
  return p;
}

}  // namespace t0mi
