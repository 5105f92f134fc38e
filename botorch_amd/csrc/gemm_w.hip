// FP64 GEMM of one 32 x 32 tile per workgroup, for products with too few rows or
// columns to fill the chip with the 128-row tiles of gemm_d.hip:
//
//   C = alpha * A op(B) + beta * C0,  A M x K, B N x K (or K x N), row-major
//
// One workgroup per tile (the tile itself: gemm_w_body.h), longest tiles first.
#include "bta_common.h"
#include "gemm.h"
#include "gemm_w.h"
#include "gemm_w_body.h"

#include <algorithm>

namespace bta {

template <int FM, int FN, int KS, int CK, int ST, bool BKN>
__global__ __launch_bounds__(64 * KS) void gemm_w_kernel(GemmArgs g, int ncu) {
  __shared__ __attribute__((aligned(1024))) unsigned char lds[w_lds<FM, FN, KS, CK, ST>()];
  gemm_w_body<FM, FN, KS, CK, ST, BKN>(g, (int)blockIdx.x, blockIdx.y, ncu, lds);
}

template <int FM, int FN, int KS, int CK, int ST>
static int w_launch(const GemmArgs& g, int batch, hipStream_t s) {
  const dim3 grid((unsigned)((int64_t)(g.M / (16 * FM)) * (g.N / (16 * FN))), (unsigned)batch);
  const dim3 th(64 * KS);
  if (g.flags & BTA_GEMM_B_KN)
    hipLaunchKernelGGL((gemm_w_kernel<FM, FN, KS, CK, ST, true>), grid, th, 0, s, g, num_cus());
  else
    hipLaunchKernelGGL((gemm_w_kernel<FM, FN, KS, CK, ST, false>), grid, th, 0, s, g, num_cus());
  BTA_LAUNCH_CHECK("gemm_w_kernel");
  return BTA_OK;
}

bool gemm_w_supported(const GemmArgs& g) {
  const uintptr_t al = (uintptr_t)g.A | (uintptr_t)g.B;
  if ((al & 15) || ((g.lda | g.ldb | g.sA | g.sB) & 1)) return false;
  if (g.M % 32 || g.N % 32 || g.K % 32 || g.M <= 0 || g.N <= 0 || g.K <= 0) return false;
  return !(g.flags & ~(BTA_GEMM_B_LOWER | BTA_GEMM_B_UPPER | BTA_GEMM_B_KN));
}

// gemm_d's 128 x 64 tiles need about two per CU; below 1.5 per CU the small tiles
// are faster (us, gemm_d / here): 1024 x 2048 (1 per CU) 138 / 101, 512 x 4096 (1)
// 257 / 190, 640 x 1024 47 / 22; at 2 per CU 2048 x 2048 takes 172 / 189.
bool gemm_w_preferred(int64_t M, int64_t N, int batch) {
  const int64_t tiles = (M + 127) / 128 * ((N + 63) / 64) * batch;
  return 2 * tiles < 3 * (int64_t)num_cus();
}

// Eight waves a tile while there is at most one tile per CU (64 x 2048: 22 us
// against 28 with four), else four and two workgroups per CU (640 x 1024: 22
// against 23).
int gemm_w(const GemmArgs& g, int batch, hipStream_t s) {
  const int64_t tiles = (int64_t)(g.M / 32) * (g.N / 32) * batch;
  if (tiles <= num_cus()) return w_launch<2, 2, 8, 16, 2>(g, batch, s);
  return w_launch<2, 2, 4, 16, 2>(g, batch, s);
}

}  // namespace bta
