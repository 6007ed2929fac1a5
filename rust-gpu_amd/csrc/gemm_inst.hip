// gemm_inst.hip — instantiates one block of gemm_variants.def for one B layout.
// Compiled eight times by the build (T0MI_PART = 0..3, T0MI_INST_NN = 0/1, with
// T0MI_TABLE_FN naming the table accessor) so the variants build in parallel.
#include "gemm_pingpong.h"
#include "t0mi_ctx.h"

#ifndef T0MI_PART
#error "T0MI_PART must be defined"
#endif
#ifndef T0MI_INST_NN
#error "T0MI_INST_NN must be defined"
#endif

namespace t0mi {

// The 256x256x64 2x4-wave configuration runs the ping-pong kernel (same
// results, bit for bit) whenever its K-granularity precondition holds.
template <int BM, int BN, int BK, int WM, int WN, int S, bool NN>
static void launch_variant(dim3 g, hipStream_t s, const GemmParams& p) {
  if constexpr (BM == 256 && BN == 256 && BK == 64 && WM == 2 && WN == 4 && S == 2) {
    if (pingpong_ok(p)) {
      hipLaunchKernelGGL((gemm_bf16_pingpong_kernel<NN, true>), g, dim3(512), 0, s, p);
      return;
    }
  }
  // Split-K's planes and outputs without an epilogue chain: kernels without its code, whose chain and biases
  // take up to twice the registers of the rest (128x128x16 on two waves: 62 VGPRs and two waves a SIMD, 234
  // and one with it).  4096x4096x512 NN, f32 out, 128x128x16: 41.0 us with the code in the kernel, 30.4
  // without; bf16 out, 128x256x32: 34.1 and 27.4; 2048x4096x1024 NN in 2 parts, 128x128x16: 55.1 and 44.2;
  // 128x4096x4096 NN in 4, 64x128x64: 14.0-14.3 and 13.9.  Planes of single waves of up to 64x64 keep the
  // one kernel: with more of them on a SIMD they run 4-6 % slower (2048x4096x1024 in 2 parts, 32x64x16 NN
  // 62.1 and 66.1 us, 64x64x16 NT 67.2 and 70.5).
  // The bf16 one stores 16 bytes at a time; a raw dispatch may bring a Y of less alignment.
  const bool planes = p.split_k > 1, aligned = !p.out_bf16 || ((uintptr_t)p.y & 15) == 0;
  if (planes ? WM * WN > 1 || BM * BN > 64 * 64 : p.epi.n == 0 && aligned) {
    if (planes || !p.out_bf16)
      hipLaunchKernelGGL((gemm_bf16_plain_kernel<BM, BN, BK, WM, WN, S, NN, kSumsF32>), g, dim3(WM * WN * 64), 0, s, p);
    else
      hipLaunchKernelGGL((gemm_bf16_plain_kernel<BM, BN, BK, WM, WN, S, NN, kSumsBf16>), g, dim3(WM * WN * 64), 0, s, p);
    return;
  }
  hipLaunchKernelGGL((gemm_bf16_kernel<BM, BN, BK, WM, WN, S, NN>), g, dim3(WM * WN * 64), 0, s, p);
}

template <int BM, int BN, int BK, int WM, int WN, int S, bool NN>
static void launch_exchange(dim3 g, hipStream_t s, const GemmParams& p, const XcdExchange& x) {
  hipLaunchKernelGGL((gemm_bf16_exchange_kernel<BM, BN, BK, WM, WN, S, NN>), g, dim3(WM * WN * 64), 0, s, p, x);
}
// Split-K summed in the launch: 64x64 tiles in two partitions (run_gemm).  The exchange costs the last
// workgroup of a tile one slot of 16 KB, the reduce launch it replaces about 1.5-2.5 us.  60 random calls
// that the ranked schedule gives that split: 1.05 times as fast (0.99 at the least: 4x480x1600), and the
// call issues one launch less (100x1000x1032: 7.4 -> 6.4 us where the host's enqueue shows).  With more to
// sum in one workgroup the reduce over the whole chip is faster: 64x64 in 4 partitions 7.6 -> 8.7 us
// (9x2432x2712), in 8 parts 8.7 -> 10.2 (12x1536x7592); 64x128 in 2 parts 11.0 -> 11.4 (2x10096x1560), in 4
// parts 9.6 -> 11.0 (8x6088x2448); 128x128 in 2 parts 16.4 -> 17.8 (68x10712x2688).
template <int BM, int BN, int BK, int WM, int WN, int S, bool NN>
static constexpr GemmExchangeFn exchange_of() {
  if constexpr (BM == 64 && BN == 64 && BK == 64 && WM * WN == 4)
    return launch_exchange<BM, BN, BK, WM, WN, S, NN>;
  else
    return nullptr;
}

#define T0MI_V(BM, BN, BK, WM, WN, S)                                                                  \
  static void launch_##BM##_##BN##_##BK##_##WM##_##WN##_##S(dim3 g, hipStream_t s, const GemmParams& p) { \
    launch_variant<BM, BN, BK, WM, WN, S, (T0MI_INST_NN != 0)>(g, s, p);                              \
  }
#if T0MI_INST_NN
#define T0MI_V_NT(BM, BN, BK, WM, WN, S)
#else
#define T0MI_V_NT(BM, BN, BK, WM, WN, S) T0MI_V(BM, BN, BK, WM, WN, S)
#endif
#include "gemm_variants.def"
#undef T0MI_V

static const GemmLaunchEntry kTable[] = {
#define T0MI_V(BM, BN, BK, WM, WN, S) \
  {BM, BN, BK, WM, WN, S, T0MI_INST_NN, launch_##BM##_##BN##_##BK##_##WM##_##WN##_##S, \
   exchange_of<BM, BN, BK, WM, WN, S, (T0MI_INST_NN != 0)>()},
#include "gemm_variants.def"
#undef T0MI_V
#undef T0MI_V_NT
};

const GemmLaunchEntry* T0MI_TABLE_FN(size_t* n) {
  *n = sizeof kTable / sizeof kTable[0];
  return kTable;
}

}  // namespace t0mi
