// Scrambled Sobol points through the inverse normal CDF, on the device.
//
// torch's SobolEngine scrambles by a lower-triangular binary matrix per dimension
// and a digital shift (both from an MT19937 stream: first the shifts' bits, least
// significant first, then the matrices, row by row, of which the part below the
// diagonal is used) and walks the points in Gray-code order.  On the CPU that is
// two serial loops over d x 30 x 30 bits and n x d points: 7 of the 9 ms that pruning
// 400 baseline points with 2048 samples took.  Here the host only draws the random
// bits (packed, one word per matrix row); the kernel scrambles the direction
// numbers of its 64 dimensions in LDS (a parity per bit) and each thread walks 16
// points of one dimension.  The points are the engine's bit for bit (the first one that
// of the default dtype float32; a caller under another one replaces it); the normal
// quantile differs from the CPU's by rounding.
#include "bta_common.h"

#include <random>

namespace bta {

constexpr int SB_BITS = 30;
constexpr int SB_DIMS = 64;   // dimensions per block
constexpr int SB_PTS = 16;    // consecutive points per thread

// cols, rows: d x 30 direction numbers and scrambling rows (bit 29 first), shift: d
__global__ __launch_bounds__(256) void sobol_normal_kernel(const uint32_t* __restrict__ cols,
                                                           const uint32_t* __restrict__ rows,
                                                           const uint32_t* __restrict__ shift,
                                                           int d, int64_t n, double eps,
                                                           double* __restrict__ out) {
  __shared__ uint32_t st[SB_DIMS][SB_BITS + 1];
  const int d0 = blockIdx.x * SB_DIMS;
  for (int e = threadIdx.x; e < SB_DIMS * SB_BITS; e += 256) {
    const int dl = e / SB_BITS, j = e % SB_BITS;
    uint32_t v = 0;
    if (d0 + dl < d) {
      const uint32_t c = cols[(int64_t)(d0 + dl) * SB_BITS + j];
      const uint32_t* r = rows + (int64_t)(d0 + dl) * SB_BITS;
      for (int p = 0; p < SB_BITS; ++p)
        v |= (uint32_t)(__popc(r[p] & c) & 1) << (SB_BITS - 1 - p);
    }
    st[dl][j] = v;
  }
  __syncthreads();
  const int dl = threadIdx.x & (SB_DIMS - 1), dim = d0 + dl;
  int64_t i = ((int64_t)blockIdx.y * 4 + (threadIdx.x >> 6)) * SB_PTS;
  if (dim >= d || i >= n) return;
  uint32_t x = shift[dim];
  for (uint32_t g = (uint32_t)i ^ ((uint32_t)i >> 1); g; g &= g - 1) x ^= st[dl][__ffs(g) - 1];
  const int64_t end = i + SB_PTS < n ? i + SB_PTS : n;
  for (;;) {
    // (the engine keeps its first point in the default dtype, float32)
    const double u = (i == 0 ? (double)(float)x : (double)x) * 0x1p-30;
    const double v = 0.5 + (1.0 - eps) * (u - 0.5);
    out[i * d + dim] = erfinv(2.0 * v - 1.0) * 1.4142135623730951;
    if (++i >= end) break;
    x ^= st[dl][__ffs((uint32_t)i) - 1];
  }
}

}  // namespace bta

extern "C" int bta_sobol_scramble(uint32_t seed, int32_t d, uint32_t* rows, uint32_t* shift) {
  using namespace bta;
  if (!rows || !shift || d < 1) {
    set_error("sobol_scramble: invalid arguments");
    return BTA_ERR_INVALID;
  }
  std::mt19937 g(seed);
  for (int i = 0; i < d; ++i) {
    uint32_t s = 0;
    for (int b = 0; b < SB_BITS; ++b) s |= (uint32_t)(g() & 1u) << b;
    shift[i] = s;
  }
  for (int64_t r = 0; r < (int64_t)d * SB_BITS; ++r) {
    const int p = (int)(r % SB_BITS);
    uint32_t row = 1u << (SB_BITS - 1 - p);  // the diagonal is one
    for (int k = 0; k < SB_BITS; ++k) {
      const uint32_t bit = (uint32_t)(g() & 1u);
      if (k < p) row |= bit << (SB_BITS - 1 - k);
    }
    rows[r] = row;
  }
  return BTA_OK;
}

extern "C" int bta_sobol_normal(const uint32_t* cols, const uint32_t* rows,
                                const uint32_t* shift, int32_t d, int64_t n, double* out,
                                bta_stream_t stream) {
  using namespace bta;
  if (!cols || !rows || !shift || !out || d < 1 || n < 1 || n > ((int64_t)1 << SB_BITS)) {
    set_error("sobol_normal: need 1 <= d and 1 <= n <= 2^30");
    return BTA_ERR_INVALID;
  }
  const int64_t gy = (n + 4 * SB_PTS - 1) / (4 * SB_PTS);
  if (gy > 65535) {
    set_error("sobol_normal: at most %d points per call", 65535 * 4 * SB_PTS);
    return BTA_ERR_UNSUPPORTED;
  }
  hipLaunchKernelGGL(sobol_normal_kernel, dim3((unsigned)((d + SB_DIMS - 1) / SB_DIMS), (unsigned)gy),
                     dim3(256), 0, (hipStream_t)stream, cols, rows, shift, d, n,
                     2.220446049250313e-16, out);
  BTA_LAUNCH_CHECK("sobol_normal_kernel");
  return BTA_OK;
}
