// CPU check of rust-gpu_amd/csrc/gemm_f32_plan.h, the rule and the global index maps of the
// one-launch f32 GEMM: for calls over its whole range, every output is stored by exactly one tile,
// the K pieces cover every K tile once and none is empty, and every 16-byte load lies inside its
// operand or is one the buffer's range check turns into zeros.
#include <cstdio>
#include <cstdlib>
#include <vector>

#include "../rust-gpu_amd/csrc/gemm_f32_plan.h"

using namespace t0mi;

static int g_fail = 0;
static long g_checks = 0;
static void check(bool ok, const char* what, int mode, unsigned m, unsigned n, unsigned k) {
  ++g_checks;
  if (!ok && ++g_fail < 20) printf("FAIL %s: mode %d m %u n %u k %u\n", what, mode, m, n, k);
}

// Loads of one operand's tile [first, first + size) over K tile kt.
static void operand(bool km, int size, uint32_t ld, int rows, int K, int first, int kt, int wanted_end, int mode,
                    unsigned m, unsigned n, unsigned k) {
  const uint64_t bytes = (uint64_t)(km ? K : rows) * ld * 4;
  const int k0 = kt * kF32Bk, ppr = (km ? size : kF32Bk) / 4, srows = km ? kF32Bk : size;
  const bool whole = k0 + kF32Bk <= K;
  for (int r = 0; r < srows; ++r)
    for (int sp = 0; sp < ppr; ++sp) {
      const uint32_t at0 = f32_piece_off(km, ld, first, rows, r, sp);
      if (at0 == kF32Oob) {  // zeros by the range check: only rows past the matrix
        check(!km && first + r >= rows && bytes < kF32MaxBytes, "row past the matrix", mode, m, n, k);
        continue;
      }
      const uint64_t off = at0 + (uint64_t)k0 * (km ? ld * 4u : 4u);
      if (km) {
        if (!whole && k0 + r >= K) continue;  // zeros by the range check
        // Columns past the matrix are read (and never stored); a piece that leaves the operand must
        // start outside of it, so that the range check drops the whole of it.
        const bool wanted = first + sp * 4 < wanted_end;
        check(off + 16 <= bytes || !wanted, "K-major load", mode, m, n, k);
        check(off < kF32MaxBytes + (1u << 20), "32-bit offset", mode, m, n, k);
      } else if (whole || (K % 4 == 0 && k0 + sp * 4 < K)) {
        check(off + 16 <= bytes, "K-contiguous load", mode, m, n, k);
      } else if (K % 4) {
        for (int j = 0; j < 4; ++j)
          if (k0 + sp * 4 + j < K) check(off + j * 4 + 4 <= bytes, "K-contiguous element", mode, m, n, k);
      }
    }
}

// Outputs: each row (and column) is stored by exactly one tile row (column); K pieces cover K once.
static void cover(const F32Plan& p, const F32Tiles& t, int mode, unsigned m, unsigned n, unsigned k) {
  for (int d = 0; d < 2; ++d) {
    const int ext = d ? (int)n : (int)m, size = d ? t.bn : t.bm, tiles = d ? (int)p.tiles_n : (int)p.tiles_m;
    std::vector<int> hit(ext, 0);
    for (int i = 0; i < tiles; ++i) {
      const int s = i * size, f = f32_tile_first(s, ext, size);
      for (int e = 0; e < size; ++e)
        if (f + e >= s && f + e < ext) ++hit[f + e];
    }
    bool ok = true;
    for (int h : hit) ok = ok && h == 1;
    check(ok, "coverage", mode, m, n, k);
  }
  check((uint64_t)p.tiles_m * p.tiles_n * p.pieces * t.bm * t.bn * 4 <= kF32SlotBytes || p.pieces == 1, "slots", mode, m,
        n, k);
  const int nkt = ((int)k + kF32Bk - 1) / kF32Bk;
  check(f32_piece_begin(0, (int)p.pieces, nkt) == 0 && f32_piece_begin((int)p.pieces, (int)p.pieces, nkt) == nkt,
        "K range", mode, m, n, k);
  for (int q = 0; q < (int)p.pieces; ++q) {
    const int b = f32_piece_begin(q, (int)p.pieces, nkt), e = f32_piece_begin(q + 1, (int)p.pieces, nkt);
    check(b < e, "empty piece", mode, m, n, k);
    check(gemm_f32_folds(t.bm, t.bn) || (uint32_t)(e - b) * kF32Bk <= kF32ChainMax, "chain", mode, m, n, k);
  }
}

// A launch that cuts K: every (tile, piece) once, slots within the tiles' own, counters apart and within
// an XCD's share.
static void workgroups(const F32Plan& p, int mode, unsigned m, unsigned n, unsigned k) {
  if (p.pieces == 1) return;
  const uint32_t nx = 8, tiles = p.tiles_m * p.tiles_n, grid = (tiles + nx - 1) / nx * nx * p.pieces;
  std::vector<int> hit(tiles * p.pieces, 0), at(tiles, -1);
  bool ok = true;
  for (uint32_t b = 0; b < grid; ++b) {
    uint32_t tile, piece, counter;
    if (!f32_workgroup(b, nx, p.pieces, tiles, &tile, &piece, &counter)) continue;
    ok = ok && tile < tiles && piece < p.pieces && counter / nx < (tiles + nx - 1) / nx;
    if (!ok) break;
    ++hit[tile * p.pieces + piece];
    ok = at[tile] < 0 || at[tile] == (int)counter;
    at[tile] = (int)counter;
  }
  for (int h : hit) ok = ok && h == 1;
  for (uint32_t i = 0; i < tiles && ok; ++i)
    for (uint32_t j = 0; j < i; ++j) ok = ok && at[i] != at[j];
  check(ok, "workgroups", mode, m, n, k);
}

// The bf16 weight's route: n and k multiples of 8 (what the entry point takes), up to 64 rows.
static void wt(unsigned m, unsigned n, unsigned k, int split, int* used) {
  const F32Plan p = wt_plan(m, n, k, 256, split);
  if (p.tile < 0) return;
  ++used[p.tile];
  const F32Tiles& t = kWtTiles[p.tile];
  check(m <= kWtMaxRows && (split || p.pieces == 1), "wt range", 3, m, n, k);
  cover(p, t, 3, m, n, k);
  workgroups(p, 3, m, n, k);
  const uint64_t bytes = (uint64_t)n * k * 2;
  for (int tn : {0, (int)p.tiles_n - 1})
    for (int kt : {0, ((int)k - 1) / kF32Bk})
      for (int r = 0; r < t.bn; ++r)
        for (int sp = 0; sp < kF32Bk / 8; ++sp) {
          const int first = f32_tile_first(tn * t.bn, (int)n, t.bn);
          const uint32_t at0 = f32_piece_off(false, k / 2, first, (int)n, r, sp);
          if (at0 == kF32Oob || kt * kF32Bk + sp * 8 >= (int)k) continue;
          check((uint64_t)at0 + (uint64_t)kt * kF32Bk * 2 + 16 <= bytes, "wt load", 3, m, n, k);
        }
}

static void one(int mode, unsigned m, unsigned n, unsigned k, int split, std::vector<int>& used) {
  const F32Plan p = f32_plan(mode, m, n, k, 256, split);
  if (p.tile < 0) {
    ++used[kF32TileCount * 4];
    return;
  }
  const F32Tiles& t = kF32Tiles[p.tile];
  int lp = 0;
  while ((1u << lp) < p.pieces) ++lp;
  ++used[p.tile * 4 + lp];
  check(split || p.pieces == 1, "pieces without the exchange", mode, m, n, k);
  cover(p, t, mode, m, n, k);
  workgroups(p, mode, m, n, k);
  const int nkt = ((int)k + kF32Bk - 1) / kF32Bk;
  // Loads: first, second last and last tile of each dimension, first and last K tiles.
  for (int kt : {0, nkt / 2, nkt - 1})
    for (int back = 0; back < 2; ++back) {
      const int tm = back == 0 ? (int)p.tiles_m - 1 : 0, tn = back == 0 ? (int)p.tiles_n - 1 : 0;
      operand(f32_a_kmajor(mode), t.bm, f32_a_kmajor(mode) ? m : k, (int)m, (int)k, f32_tile_first(tm * t.bm, (int)m, t.bm),
              kt, (int)m, mode, m, n, k);
      operand(f32_b_kmajor(mode), t.bn, f32_b_kmajor(mode) ? n : k, (int)n, (int)k, f32_tile_first(tn * t.bn, (int)n, t.bn),
              kt, (int)n, mode, m, n, k);
    }
}

// Calls near the line whose measured times are more than 1.15 apart: the faster route.
static void routes() {
  const struct {
    int mode;
    unsigned m, n, k;
    bool one_launch;
  } c[] = {{F32_DATA, 696, 192, 8128, false},   {F32_DATA, 564, 344, 7232, false},  {F32_FORWARD, 927, 320, 7232, false},
           {F32_DATA, 653, 384, 7424, false},   {F32_FORWARD, 886, 216, 7408, false}, {F32_FORWARD, 622, 328, 7984, false},
           {F32_DATA, 91, 1280, 6784, true},    {F32_FORWARD, 79, 1408, 4544, true}, {F32_DATA, 222, 2048, 6912, true},
           {F32_FORWARD, 69, 3800, 5672, true}, {F32_FORWARD, 436, 417, 6683, true}};
  for (const auto& x : c)
    check((f32_plan(x.mode, x.m, x.n, x.k, 256, true).tile >= 0) == x.one_launch, "route", x.mode, x.m, x.n, x.k);
}

int main() {
  routes();
  std::vector<int> used(kF32TileCount * 4 + 1, 0);
  srand(1);
  const unsigned edge[] = {1, 2, 3, 4, 5, 7, 8, 15, 16, 31, 32, 33, 63, 64, 65, 66, 100, 127, 128, 129, 255, 333, 1000, 4096};
  for (int mode = 0; mode < 3; ++mode)
    for (int split = 0; split < 2; ++split) {
      for (unsigned m : edge)
        for (unsigned n : edge)
          for (unsigned k : edge) one(mode, m, n, k, split, used);
      for (int i = 0; i < 400; ++i) {
        auto r = [] { return 1u + (unsigned)rand() % (1u << (1 + rand() % 14)); };
        const unsigned m = r(), n = r(), k = r();
        one(mode, m, n, k, split, used);
      }
    }
  int wt_used[kWtTileCount] = {};
  for (int split = 0; split < 2; ++split)
    for (int i = 0; i < 4000; ++i)
      wt(1 + (unsigned)rand() % 70, 8 * (1 + (unsigned)rand() % (1u << (1 + rand() % 11))),
         8 * (1 + (unsigned)rand() % (1u << (1 + rand() % 10))), split, wt_used);
  for (int i = 0; i < kWtTileCount; ++i) g_fail += wt_used[i] == 0;
  for (int i = 0; i < kF32TileCount; ++i)
    printf("%dx%d pieces 1/2/4/8: %d %d %d %d\n", kF32Tiles[i].bm, kF32Tiles[i].bn, used[i * 4], used[i * 4 + 1],
           used[i * 4 + 2], used[i * 4 + 3]);
  printf("two passes: %d\n%ld checks, %d failures\n", used[kF32TileCount * 4], g_checks, g_fail);
  for (int i = 0; i < kF32TileCount; ++i) g_fail += used[i * 4] == 0;  // every tile is reachable
  return g_fail != 0;
}
