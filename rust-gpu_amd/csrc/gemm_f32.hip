// gemm_f32.hip — launches of the one-launch f32-operand GEMM (gemm_f32.h) for the Ignis matmul
// (src/ignis/ops/bf16_matmul.rs:33-316).
#include "gemm_f32.h"

#include <string.h>

#include "t0mi_ctx.h"

namespace t0mi {

namespace {

template <int I, bool AK, bool BKM>
void launch(const GemmF32Params& p, uint32_t grid, hipStream_t s) {
  constexpr int BM = kF32Tiles[I].bm, BN = kF32Tiles[I].bn, G = kF32Tiles[I].groups;
  constexpr int WM = I == 0 ? 1 : I == 3 ? 4 : 2, WN = I < 2 ? 1 : I == 4 ? 4 : 2;  // 8 waves with G
  hipLaunchKernelGGL((gemm_f32_kernel<BM, BN, kF32Bk, WM, WN, G, 2, AK, BKM>), dim3(grid), dim3(WM * WN * G * 64), 0,
                     s, p);
}

template <bool AK, bool BKM>
void launch_tile(int tile, const GemmF32Params& p, uint32_t grid, hipStream_t s) {
  switch (tile) {
    case 0: launch<0, AK, BKM>(p, grid, s); break;
    case 1: launch<1, AK, BKM>(p, grid, s); break;
    case 2: launch<2, AK, BKM>(p, grid, s); break;
    case 3: launch<3, AK, BKM>(p, grid, s); break;
    default: launch<4, AK, BKM>(p, grid, s); break;
  }
}

void launch_wt(int tile, const GemmF32Params& p, uint32_t grid, hipStream_t s) {
  constexpr const F32Tiles &T0 = kWtTiles[0], &T1 = kWtTiles[1];
  if (tile == 0)
    hipLaunchKernelGGL((gemm_f32_kernel<T0.bm, T0.bn, kF32Bk, 1, 2, T0.groups, 2, false, false, true>), dim3(grid),
                       dim3(512), 0, s, p);
  else
    hipLaunchKernelGGL((gemm_f32_kernel<T1.bm, T1.bn, kF32Bk, 2, 2, T1.groups, 2, false, false, true>), dim3(grid),
                       dim3(512), 0, s, p);
}

// Fills the parameters of a planned call and *grid.  1: the call takes the other route (an operand
// overlaps Y, which that route reads whole before Y is written; or the exchange cannot be had now).
int set_up(t0mi_ctx* ctx, const F32Plan& plan, int b_size, uint64_t a, uint64_t b, uint64_t y, uint32_t m, uint32_t n,
           uint32_t k, GemmF32Params* p, uint32_t* grid) {
  if (plan.tile < 0) return 1;
  const uint64_t a_bytes = (uint64_t)m * k * 4, b_bytes = (uint64_t)k * n * b_size, y_bytes = (uint64_t)m * n * 4;
  if (ranges_meet(a, a_bytes, y, y_bytes) || ranges_meet(b, b_bytes, y, y_bytes)) return 1;
  memset(p, 0, sizeof *p);
  p->a = (const float*)a;
  p->b = (const void*)b;
  p->y = (float*)y;
  p->M = m;
  p->N = n;
  p->K = k;
  p->a_bytes = (uint32_t)a_bytes;
  p->b_bytes = (uint32_t)b_bytes;
  p->tiles_m = plan.tiles_m;
  p->tiles_n = plan.tiles_n;
  p->pieces = plan.pieces;
  *grid = plan.tiles_m * plan.tiles_n;
  // The slots are made by the first call of this route, split or not: what a later call may do under
  // capture depends on a call before it, not on that call's sizes.
  bool ok = false;
  if (int rc = xk_prepare(ctx, *grid, kF32SlotBytes, &p->x, &ok, true)) return rc;
  if (plan.pieces > 1) {
    if (!ok) return 1;
    *grid = (*grid + p->x.nx - 1) / p->x.nx * p->x.nx * plan.pieces;
  }
  return T0MI_OK;
}

int launched() {
  const hipError_t e = hipGetLastError();
  return e == hipSuccess ? T0MI_OK : set_error(T0MI_ERR_HIP, "f32 GEMM launch: %s", hipGetErrorString(e));
}

}  // namespace

int run_gemm_f32(t0mi_ctx* ctx, int mode, uint64_t a, uint64_t b, uint64_t y, uint32_t m, uint32_t n, uint32_t k) {
  if (ctx->null_backend) return 1;
  const F32Plan plan = f32_plan(mode, m, n, k, (uint32_t)ctx->cu_count, ctx->xk_nx > 0);
  GemmF32Params p;
  uint32_t grid;
  if (int rc = set_up(ctx, plan, 4, a, b, y, m, n, k, &p, &grid)) return rc;
  p.lda = f32_a_kmajor(mode) ? m : k;
  p.ldb = f32_b_kmajor(mode) ? n : k;
  switch (mode) {
    case F32_FORWARD: launch_tile<false, true>(plan.tile, p, grid, ctx->stream); break;
    case F32_DATA: launch_tile<false, false>(plan.tile, p, grid, ctx->stream); break;
    default: launch_tile<true, true>(plan.tile, p, grid, ctx->stream); break;
  }
  return launched();
}

int run_gemm_wt(t0mi_ctx* ctx, uint64_t x, uint64_t wt, uint64_t y, uint32_t m, uint32_t n, uint32_t k) {
  if (ctx->null_backend) return 1;
  const F32Plan plan = wt_plan(m, n, k, (uint32_t)ctx->cu_count, ctx->xk_nx > 0);
  GemmF32Params p;
  uint32_t grid;
  if (int rc = set_up(ctx, plan, 2, x, wt, y, m, n, k, &p, &grid)) return rc;
  p.lda = k;
  p.ldb = k;
  launch_wt(plan.tile, p, grid, ctx->stream);
  return launched();
}

}  // namespace t0mi
