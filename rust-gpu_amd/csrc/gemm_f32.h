// gemm_f32.h — Y = bf16(A) . bf16(B) with f32 operands and f32 output in one launch (gfx950).
//
// The Ignis matmul (src/ignis/ops/bf16_matmul.rs:33-316) has f32 tensors on both sides of a
// bf16 product: forward Y = X . W, data gradient dX = dY . W^T, weight gradient
// dW = X^T . dY.  A conversion pass per operand (and, for X^T, a transposing one), the GEMM,
// its split-K reduce and an unpad pass are four to six launches whose fixed cost exceeds the
// product's own time up to mid-sized layers.  Here every workgroup loads its f32 tiles into
// registers, rounds them (RNE, v_cvt_pk_bf16_f32, the same rounding as the conversion pass)
// on the way into LDS and multiplies with v_mfma_f32_32x32x16_bf16.
//
//   * An operand is either K-contiguous (rows of the f32 matrix are rows / columns of the
//     product: X and dY on the left, W^T) or K-major (rows of the f32 matrix are K: W and dY
//     on the right, X^T on the left).  K-contiguous tiles land in LDS as [rows][BK] and are
//     read with ds_read_b128; K-major tiles land as loaded, [BK][columns], and the operand is
//     formed by ds_read_b64_tr_b16.  No transpose pass for any of the three products.
//   * Loads are 16 bytes per lane through a buffer resource, so rows of any length (only
//     4-byte aligned) are taken as they are; past the end of K they read zero through the
//     resource's range check.
//   * A workgroup's G wave groups take every G-th K tile, each with its own LDS buffers, and
//     their sums meet in LDS at the end in group order: a fixed order, so results do not
//     depend on timing.  D K tiles per group are in flight in registers while another is multiplied
//     from LDS.
//   * Where the tiles are fewer than the CUs, K is also cut over `pieces` workgroups per tile in
//     the same launch; their sums are exchanged through memory (xcd_exchange.h) and added in piece
//     order by the workgroup that arrives last.
//   * The right operand may also be bf16 and K-contiguous: the inference layer on its cached weight
//     (bf16_matmul.rs:99-134).
//   * A tile that would end past the matrix starts earlier instead (it overlaps its neighbour,
//     whose rows and columns it does not store), so no load needs a column mask.
//
// What bounds it: the CU's load path.  A further K tile's f32 pieces enter a CU at 107-112 GB/s whatever the
// tile and however many are in flight (two K tiles per group or four: the same times), so the time
// is the operand bytes per CU, (bm + bn) * 4 * K for each of its tiles, over that rate, plus about
// 4 us; hence larger tiles as soon as they still give every CU one, and K cut over workgroups where
// they do not.  Large products pay that twice over (f32 pieces are twice the bf16 bytes, read once
// per tile row and column), and the conversion passes win: f32_plan (gemm_f32_plan.h) draws the line.
// Measured, forward + data + weight of one layer, before (conversion passes, GEMM, reduce, unpad) and
// now: 512 tokens, 1024 -> 4096: 66.8 -> 49.2 us; 333 tokens, 1100 -> 770: 56.1 -> 29.6 us; forward
// alone, 16 x 4096 x 4096: 27.9 -> 17.2 us; inference layer, 7 x 11008 x 2048: 12.7 -> 10.6 us.  The
// error against 64-bit sums is the smaller one (1.9e-7 -> 1.2e-7 relative on the first): K is summed in chains of at most 1024.
#pragma once
#include <type_traits>

#include "gemm_bf16_kernel.h"
#include "gemm_f32_plan.h"
#include "xcd_exchange.h"

namespace t0mi {

struct GemmF32Params {
  const float* a;  // K-contiguous: [M][lda]; K-major: [K][lda], M columns
  const void* b;   // K-contiguous: [N][ldb]; K-major: [K][ldb], N columns; f32 or bf16
  float* y;        // [M][N]
  uint32_t M, N, K, lda, ldb;
  uint32_t a_bytes, b_bytes;  // extent of each operand (below 2 GiB)
  uint32_t tiles_m, tiles_n;
  uint32_t pieces;  // K pieces per tile (workgroups); above 1 the exchange below is used
  XcdExchange x;
};

// One operand's tile: ROWS rows (or columns) of the product by BK of K, loaded by NT threads as
// NP 16-byte pieces each; KM: K-major.
template <int ROWS_, int BK_, int NT, bool KM_>
struct F32Tile {
  static constexpr int ROWS = ROWS_, BK = BK_;
  static constexpr bool KM = KM_;
  static constexpr int PPR = (KM ? ROWS : BK) / 4;   // pieces per source row
  static constexpr int NP = ROWS * BK / 4 / NT;      // pieces per thread
  static constexpr int RSTEP = NT / PPR;             // source rows between a thread's pieces
  static constexpr int KC = BK / 8, NC = ROWS / 8;   // 16-byte bf16 chunks per LDS row
  static constexpr int ELEMS = ROWS * BK;
  static_assert(NP * NT * 4 == ROWS * BK && NT % PPR == 0, "whole pieces per thread");

  __amdgpu_buffer_rsrc_t rs;
  int sr, sp;          // the thread's first source row and its piece in a row
  uint32_t off[NP];    // byte offset of each piece at K = 0
  uint32_t kstep;      // bytes per unit of K

  // `first`: the tile's first row (column) of the product; `rows`: the matrix's.
  __device__ __forceinline__ void init(const void* base, uint32_t bytes, uint32_t ld, int first, int rows, int t) {
    rs = __builtin_amdgcn_make_buffer_rsrc((void*)base, (short)0, (int)bytes, 0x00020000);
    sr = t / PPR;
    sp = t % PPR;
    kstep = KM ? ld * 4u : 4u;
#pragma unroll
    for (int i = 0; i < NP; ++i) off[i] = f32_piece_off(KM, ld, first, rows, sr + i * RSTEP, sp);
  }
  // K tile starting at k0, whole.
  __device__ __forceinline__ void load_full(int k0, f32x4* v) const {
    const int so = __builtin_amdgcn_readfirstlane((int)((uint32_t)k0 * kstep));
#pragma unroll
    for (int i = 0; i < NP; ++i)
      v[i] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(rs, (int)off[i], so, 0));
  }
  // A K tile that K cuts, or that starts past it: zeros there.  A K-contiguous piece that K cuts
  // (K % 4 != 0) is loaded element by element.
  __device__ __forceinline__ void load_cut(int k0, int K, f32x4* v) const {
    const uint32_t ko = (uint32_t)k0 * kstep;
    if (!KM && (K & 3)) {
#pragma unroll
      for (int i = 0; i < NP; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const uint32_t o = k0 + sp * 4 + j < K ? off[i] + ko + (uint32_t)j * 4u : kF32Oob;
          v[i][j] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rs, (int)o, 0, 0));
        }
    } else {
#pragma unroll
      for (int i = 0; i < NP; ++i) {
        const int k = KM ? k0 + sr + i * RSTEP : k0 + sp * 4;
        v[i] = __builtin_bit_cast(
            f32x4, __builtin_amdgcn_raw_buffer_load_b128(rs, (int)(k < K ? off[i] + ko : kF32Oob), 0, 0));
      }
    }
  }
  // LDS element of column `col` (a multiple of 4) of K row k.  Rows of 32 columns need no swizzle:
  // the 4 rows x 32 columns of a half-wave's transpose read are 256 contiguous bytes.
  __device__ __forceinline__ static int km_elem(int k, int col) {
    if constexpr (NC >= 8)
      return nn_elem<NC>(k, col);
    else
      return k * ROWS + col;
  }
  // The pieces, rounded to bf16, into the LDS tile.
  __device__ __forceinline__ void store_lds(uint16_t* lds, const f32x4* v) const {
#pragma unroll
    for (int i = 0; i < NP; ++i) {
      const int r = sr + i * RSTEP;
      const int e = KM ? km_elem(r, sp * 4) : kc_slot<KC>(r, sp >> 1) * 8 + (sp & 1) * 4;
      u32x2 o;
      o.x = pack_bf16x2(v[i].x, v[i].y);
      o.y = pack_bf16x2(v[i].z, v[i].w);
      *(u32x2*)(lds + e) = o;
    }
  }
  // The MFMA operand of rows (columns) r0 .. r0+31 at k-step ks: lane l holds row l % 32,
  // K 8 * (l / 32) .. +7 of the step.
  __device__ __forceinline__ static bf16x8 frag(const uint16_t* lds, int r0, int ks, int lane) {
    if constexpr (!KM) {
      return *(const bf16x8*)(lds + kc_slot<KC>(r0 + (lane & 31), ks * 2 + (lane >> 5)) * 8);
    } else {
      const int tg = lane >> 4, ti = lane & 15;
      const int krow = ks * 16 + 8 * (tg >> 1) + (ti >> 2), col = r0 + 16 * (tg & 1) + 4 * (ti & 3);
      i16x4 h[2];
#pragma unroll
      for (int j = 0; j < 2; ++j)
        h[j] = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
            (__attribute__((address_space(3))) i16x4*)(lds + km_elem(krow + 4 * j, col)));
      u32x4 u;
      u.x = (uint32_t)(uint16_t)h[0].x | ((uint32_t)(uint16_t)h[0].y << 16);
      u.y = (uint32_t)(uint16_t)h[0].z | ((uint32_t)(uint16_t)h[0].w << 16);
      u.z = (uint32_t)(uint16_t)h[1].x | ((uint32_t)(uint16_t)h[1].y << 16);
      u.w = (uint32_t)(uint16_t)h[1].z | ((uint32_t)(uint16_t)h[1].w << 16);
      return __builtin_bit_cast(bf16x8, u);
    }
  }
};

// The same for a bf16 operand, K-contiguous (the cached weight of the inference layer, used in
// place): pieces of 8 elements go to LDS as they are.  K is a multiple of 8.
template <int ROWS_, int BK_, int NT>
struct Bf16Tile {
  static constexpr int ROWS = ROWS_, BK = BK_;
  static constexpr int PPR = BK / 8, NP = ROWS * BK / 8 / NT, RSTEP = NT / PPR, KC = BK / 8;
  static constexpr int ELEMS = ROWS * BK;
  static_assert(NP * NT * 8 == ROWS * BK && NT % PPR == 0, "whole pieces per thread");

  __amdgpu_buffer_rsrc_t rs;
  int sr, sp;
  uint32_t off[NP];

  __device__ __forceinline__ void init(const void* base, uint32_t bytes, uint32_t ld, int first, int rows, int t) {
    rs = __builtin_amdgcn_make_buffer_rsrc((void*)base, (short)0, (int)bytes, 0x00020000);
    sr = t / PPR;
    sp = t % PPR;
#pragma unroll
    for (int i = 0; i < NP; ++i) off[i] = f32_piece_off(false, ld / 2, first, rows, sr + i * RSTEP, sp);
  }
  __device__ __forceinline__ void load_full(int k0, f32x4* v) const {
    const int so = __builtin_amdgcn_readfirstlane(k0 * 2);
#pragma unroll
    for (int i = 0; i < NP; ++i)
      v[i] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(rs, (int)off[i], so, 0));
  }
  __device__ __forceinline__ void load_cut(int k0, int K, f32x4* v) const {
#pragma unroll
    for (int i = 0; i < NP; ++i) {
      const uint32_t o = k0 + sp * 8 < K ? off[i] + (uint32_t)k0 * 2u : kF32Oob;
      v[i] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(rs, (int)o, 0, 0));
    }
  }
  __device__ __forceinline__ void store_lds(uint16_t* lds, const f32x4* v) const {
#pragma unroll
    for (int i = 0; i < NP; ++i) *(f32x4*)(lds + kc_slot<KC>(sr + i * RSTEP, sp) * 8) = v[i];
  }
  __device__ __forceinline__ static bf16x8 frag(const uint16_t* lds, int r0, int ks, int lane) {
    return *(const bf16x8*)(lds + kc_slot<KC>(r0 + (lane & 31), ks * 2 + (lane >> 5)) * 8);
  }
};

// BM x BN of Y per workgroup of G groups of WM x WN waves.  AK / BKM: the operand is K-major;
// B16: the right operand is bf16.
template <int BM, int BN, int BK, int WM, int WN, int G, int D, bool AK, bool BKM, bool B16 = false>
__global__ __launch_bounds__(WM* WN* G * 64) void gemm_f32_kernel(GemmF32Params p) {
  constexpr int GT = WM * WN * 64;  // threads per group
  constexpr int TM = BM / WM, TN = BN / WN, FM = TM / 32, FN = TN / 32, KS = BK / 16;
  constexpr bool FOLD = gemm_f32_folds(BM, BN);
  constexpr int kFoldTiles = 512 / BK;
  using TA = F32Tile<BM, BK, GT, AK>;
  using TB = std::conditional_t<B16, Bf16Tile<BN, BK, GT>, F32Tile<BN, BK, GT, BKM>>;
  constexpr int STAGE = TA::ELEMS + TB::ELEMS;  // bf16 elements of one LDS stage
  constexpr int LDO = BN + 4;                   // f32 row length of the output block in LDS
  constexpr int RING_BYTES = G * 2 * STAGE * 2, OUT_BYTES = G * BM * LDO * 4;
  __shared__ __attribute__((aligned(1024))) char smem[RING_BYTES > OUT_BYTES ? RING_BYTES : OUT_BYTES];

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const int grp = wave / (WM * WN), w = wave % (WM * WN);
  const int wm = w / WN, wn = w % WN;
  const int t = (int)threadIdx.x % GT;
  uint16_t* ring = (uint16_t*)smem + grp * 2 * STAGE;

  // Workgroup -> (tile, K piece).  Neighbouring tiles share an XCD (and its L2).
  int tm, tn, part;
  uint32_t tile = 0, piece = 0, counter = 0;
  if (p.pieces == 1) {
    tile_coords_of(p.tiles_m, p.tiles_n, 1, tm, tn, part);
  } else {
    xk_check_placement(p.x);
    const uint32_t tiles = p.tiles_m * p.tiles_n;
    if (!f32_workgroup(blockIdx.x, p.x.nx, p.pieces, tiles, &tile, &piece, &counter)) return;
    tile_coords_lin(tile, tiles, p.tiles_m, p.tiles_n, 0, tm, tn, part);
  }
  const int M = (int)p.M, N = (int)p.N;
  const int nkt = ((int)p.K + BK - 1) / BK;  // K tiles, cut evenly over the pieces
  const int kb = f32_piece_begin((int)piece, (int)p.pieces, nkt);
  const int ke = f32_piece_begin((int)piece + 1, (int)p.pieces, nkt);
  const int K = min((int)p.K, ke * BK);  // end of this piece's K range
  const int ms = tm * BM, ns = tn * BN;  // first row / column stored
  const int m0 = f32_tile_first(ms, M, BM), n0 = f32_tile_first(ns, N, BN);
  TA ta;
  TB tb;
  ta.init(p.a, p.a_bytes, p.lda, m0, M, t);
  tb.init(p.b, p.b_bytes, p.ldb, n0, N, t);

  f32x16 acc[FN][FM] = {}, sum[FN][FM] = {};
  // Every kFoldTiles K tiles the running sums are added to a second set: the rounding error of a
  // long K range then grows with its pieces, as a split-K sum's does.
  auto fold = [&]() {
#pragma unroll
    for (int fn = 0; fn < FN; ++fn)
#pragma unroll
      for (int fm = 0; fm < FM; ++fm) {
        sum[fn][fm] += acc[fn][fm];
        acc[fn][fm] = f32x16{};
      }
  };

  const int nit = (ke - kb + G - 1) / G;  // group g multiplies K tiles kb + g, kb + g + G, ...
  f32x4 va[D][TA::NP], vb[D][TB::NP];
  // K tile i of the group into register set s; CUT: K may end in it or before it.
  auto load = [&](int i, auto set_c, auto cut_c) {
    constexpr int s = decltype(set_c)::value % D;
    const int k0 = (kb + i * G + grp) * BK;
    if (!decltype(cut_c)::value || k0 + BK <= K) {
      ta.load_full(k0, va[s]);
      tb.load_full(k0, vb[s]);
    } else {
      ta.load_cut(k0, K, va[s]);
      tb.load_cut(k0, K, vb[s]);
    }
  };
  // Register set s into its LDS stage.
  auto store = [&](auto set_c) {
    constexpr int s = decltype(set_c)::value % D;
    ta.store_lds(ring + s % 2 * STAGE, va[s]);
    tb.store_lds(ring + s % 2 * STAGE + TA::ELEMS, vb[s]);
  };
  auto multiply = [&](auto set_c) {
    const uint16_t* As = ring + decltype(set_c)::value % 2 * STAGE;
    const uint16_t* Bs = As + TA::ELEMS;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      bf16x8 xa[FM], xb[FN];
#pragma unroll
      for (int fm = 0; fm < FM; ++fm) xa[fm] = TA::frag(As, wm * TM + fm * 32, ks, lane);
#pragma unroll
      for (int fn = 0; fn < FN; ++fn) xb[fn] = TB::frag(Bs, wn * TN + fn * 32, ks, lane);
#pragma unroll
      for (int fn = 0; fn < FN; ++fn)
#pragma unroll
        for (int fm = 0; fm < FM; ++fm)
          acc[fn][fm] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(xb[fn], xa[fm], acc[fn][fm], 0, 0, 0);
    }
  };
  // LDS writes and reads of this wave done, then the workgroup barrier (loads stay in flight).
  auto barrier = [&]() {
    wait_lgkmcnt0();
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
  };
  // Tile i of a group sits in register set i % D and LDS stage i % 2: tile i + 1 goes from
  // registers to LDS while tile i is multiplied, and tile i + 1 + D takes its registers.
  using Cut = std::integral_constant<bool, true>;
  using Whole = std::integral_constant<bool, false>;
  static_for<D>([&](auto sc) { load(decltype(sc)::value, sc, Cut{}); });
  store(std::integral_constant<int, 0>{});
  load(D, std::integral_constant<int, 0>{}, Cut{});
  barrier();
  auto iteration = [&](int i, auto sc, auto cut_c) {  // i % D == sc
    constexpr int s = decltype(sc)::value;
    using Next = std::integral_constant<int, s + 1>;
    store(Next{});
    load(i + 1 + D, Next{}, cut_c);
    multiply(sc);
    barrier();
  };
  const int nfull = (K / BK - kb) / G;  // tiles i < nfull are whole in every group
  int i = 0;
  while (i + 2 * D < nfull) {
    const int stop = FOLD ? min(nfull - 2 * D, i + kFoldTiles) : nfull - 2 * D;
    for (; i < stop; i += D) static_for<D>([&](auto sc) { iteration(i + decltype(sc)::value, sc, Whole{}); });
    if (FOLD) fold();
  }
  for (; i < nit; i += D)
    static_for<D>([&](auto sc) {
      if (i + decltype(sc)::value < nit) iteration(i + decltype(sc)::value, sc, Cut{});
    });
  if (FOLD) fold();

  // Lane l of block (fn, fm) holds row fm*32 + (l & 31), columns fn*32 + 8*g + 4*(l >> 5) + 0..3.
  // Every group's block goes to LDS (the ring is idle after the last barrier), then the
  // workgroup sums them in group order and stores whole row segments.
  float* out = (float*)smem;
#pragma unroll
  for (int fn = 0; fn < FN; ++fn)
#pragma unroll
    for (int fm = 0; fm < FM; ++fm)
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        const int r = wm * TM + fm * 32 + (lane & 31), c = wn * TN + fn * 32 + g * 8 + (lane >> 5) * 4;
        const f32x16& x = FOLD ? sum[fn][fm] : acc[fn][fm];
        *(f32x4*)(out + (grp * BM + r) * LDO + c) = f32x4{x[g * 4], x[g * 4 + 1], x[g * 4 + 2], x[g * 4 + 3]};
      }
  barrier();
  constexpr int PR = BN / 4, ROWS_PER = GT * G / PR < BM ? GT * G / PR : BM, NOUT = BM / ROWS_PER;
  static_assert(NOUT * ROWS_PER == BM && GT * G % PR == 0, "whole rows per pass");
  const bool act = (int)threadIdx.x < ROWS_PER * PR;  // small tiles have fewer pieces than threads
  const int r0 = act ? (int)threadIdx.x / PR : 0, c = ((int)threadIdx.x % PR) * 4;
  f32x4 s[NOUT];
#pragma unroll
  for (int j = 0; j < NOUT; ++j) {
    const int r = r0 + j * ROWS_PER;
    s[j] = *(const f32x4*)(out + r * LDO + c);
#pragma unroll
    for (int g = 1; g < G; ++g) s[j] += *(const f32x4*)(out + (g * BM + r) * LDO + c);
  }
  if (p.pieces > 1) {
    constexpr uint32_t SLOT = (uint32_t)(BM * BN * 4);
    const __amdgpu_buffer_rsrc_t sl =
        xk_slots(p.x.part + (size_t)tile * p.pieces * (BM * BN), p.pieces * SLOT);
    const uint32_t o = (uint32_t)((r0 * BN + c) * 4);
#pragma unroll
    for (int j = 0; j < NOUT; ++j)
      if (act) xk_store(sl, piece * SLOT + o + (uint32_t)(j * ROWS_PER * BN * 4), __builtin_bit_cast(xk_f32x4, s[j]));
    if (!xk_arrive(p.x, counter, p.pieces)) return;
#pragma unroll
    for (int j = 0; j < NOUT; ++j) s[j] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    for (uint32_t q0 = 0; q0 < p.pieces; q0 += 2) {  // pieces are a power of two
      f32x4 u[2][NOUT];
#pragma unroll
      for (int q = 0; q < 2; ++q)
#pragma unroll
        for (int j = 0; j < NOUT; ++j)
          u[q][j] = __builtin_bit_cast(
              f32x4, xk_load(sl, (q0 + (uint32_t)q) * SLOT + o + (uint32_t)(j * ROWS_PER * BN * 4)));
#pragma unroll
      for (int j = 0; j < NOUT; ++j) s[j] = s[j] + u[0][j] + u[1][j];
    }
    xk_reset(p.x, counter);
  }
  const bool whole = n0 == ns && n0 + BN <= N;  // every column is this tile's and inside N
#pragma unroll
  for (int j = 0; j < NOUT; ++j) {
    const int r = m0 + r0 + j * ROWS_PER;
    if (!act || r < ms || r >= M) continue;
    float* d = p.y + (size_t)r * N + n0 + c;
    if (whole) {
      *(f32x4_a4*)d = s[j];
    } else {
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (n0 + c + e >= ns && n0 + c + e < N) d[e] = s[j][e];
    }
  }
}

}  // namespace t0mi
