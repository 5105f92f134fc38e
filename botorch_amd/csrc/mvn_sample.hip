// Reparameterised samples of many small multivariate normals and their adjoint.
//
//   out[s][b][i] = mean[b][i] + sum_{j <= i} L[b][i][j] z[s][b][j]
//   dL[b][i][j] = sum_s g[s][b][i] z[s][b][j] (j <= i),  dmean[b][i] = sum_s g[s][b][i]
//
// for m <= 16 points per element.  The GEMM these replace at that size padded every
// element to 64 x 64 x 64 and needed a dozen small launches around it to pad,
// expand, transpose and add (256 elements of 4 points, 64 samples: 14 launches and
// about 110 us forward, 10 and 80 us backward).  The base samples are read through
// their strides, so samples shared by all elements are not copied per element.
#include "bta_common.h"

namespace bta {

constexpr int MS_MAX_M = 16;

// one output per thread, in the order of out: neighbouring threads share the
// element's rows of L and its base samples
__global__ __launch_bounds__(256) void mvn_sample_kernel(const double* __restrict__ mean,
                                                         const double* __restrict__ L,
                                                         const double* __restrict__ z, int64_t zs,
                                                         int64_t zb, int64_t S, int64_t nb, int m,
                                                         double* __restrict__ out) {
  const int64_t total = S * nb * m;
  for (int64_t e = (int64_t)blockIdx.x * 256 + threadIdx.x; e < total;
       e += (int64_t)gridDim.x * 256) {
    const int64_t row = e / m, s = row / nb, b = row - s * nb;
    const int i = (int)(e - row * m);
    const double* l = L + (b * m + i) * m;
    const double* x = z + s * zs + b * zb;
    double v = 0.0;
    for (int j = 0; j <= i; ++j) v = fma(l[j], x[j], v);
    out[e] = v + mean[b * m + i];
  }
}

// One workgroup per element.  The m (m + 1) / 2 products and m sums of the element
// go to as many threads, repeated G times over interleaved samples; the G shares
// are added in order.
__global__ __launch_bounds__(256) void mvn_sample_backward_kernel(
    const double* __restrict__ g, const double* __restrict__ z, int64_t zs, int64_t zb, int64_t S,
    int64_t nb, int m, double* __restrict__ dmean, double* __restrict__ dL) {
  __shared__ double red[256];
  const int64_t b = blockIdx.x;
  const int np = m * (m + 1) / 2, per = np + m, G = 256 / per;
  const int t = threadIdx.x, item = t % per, share = t / per;
  int i = 0, j = -1;  // j < 0: the sum over the samples
  if (item < np) {
    while ((i + 1) * (i + 2) / 2 <= item) ++i;
    j = item - i * (i + 1) / 2;
  } else {
    i = item - np;
  }
  double v = 0.0;
  if (share < G)
    for (int64_t s = share; s < S; s += G) {
      const double gv = g[(s * nb + b) * m + i];
      v = j < 0 ? v + gv : fma(gv, z[s * zs + b * zb + j], v);
    }
  red[t] = v;
  __syncthreads();
  if (t < per) {
    double sum = red[t];
    for (int k = 1; k < G; ++k) sum += red[k * per + t];
    if (j < 0) {
      dmean[b * m + i] = sum;
    } else {
      dL[(b * m + i) * m + j] = sum;
      if (j < i) dL[(b * m + j) * m + i] = 0.0;
    }
  }
}

static int mvn_check(const char* what, int64_t S, int64_t nb, int m) {
  if (m < 1 || m > MS_MAX_M || S < 0 || nb < 0 || nb > (1 << 30) || S > ((int64_t)1 << 32)) {
    set_error("%s: need 1 <= m <= %d", what, MS_MAX_M);
    return BTA_ERR_UNSUPPORTED;
  }
  return BTA_OK;
}

}  // namespace bta

extern "C" int bta_mvn_sample(const double* mean, const double* L, const double* z, int64_t z_s,
                              int64_t z_b, int64_t S, int64_t batch, int32_t m, double* out,
                              bta_stream_t stream) {
  using namespace bta;
  int rc = mvn_check("mvn_sample", S, batch, m);
  if (rc) return rc;
  if (S == 0 || batch == 0) return BTA_OK;
  if (!mean || !L || !z || !out) {
    set_error("mvn_sample: null pointer");
    return BTA_ERR_INVALID;
  }
  const int64_t blocks = (S * batch * m + 255) / 256;
  hipLaunchKernelGGL(mvn_sample_kernel, dim3((unsigned)(blocks < 65536 ? blocks : 65536)),
                     dim3(256), 0, (hipStream_t)stream, mean, L, z, z_s, z_b, S, batch, m, out);
  BTA_LAUNCH_CHECK("mvn_sample_kernel");
  return BTA_OK;
}

extern "C" int bta_mvn_sample_backward(const double* g, const double* z, int64_t z_s, int64_t z_b,
                                       int64_t S, int64_t batch, int32_t m, double* dmean,
                                       double* dL, bta_stream_t stream) {
  using namespace bta;
  int rc = mvn_check("mvn_sample_backward", S, batch, m);
  if (rc) return rc;
  if (batch == 0) return BTA_OK;
  if (!g || !z || !dmean || !dL) {
    set_error("mvn_sample_backward: null pointer");
    return BTA_ERR_INVALID;
  }
  hipLaunchKernelGGL(mvn_sample_backward_kernel, dim3((unsigned)batch), dim3(256), 0,
                     (hipStream_t)stream, g, z, z_s, z_b, S, batch, m, dmean, dL);
  BTA_LAUNCH_CHECK("mvn_sample_backward_kernel");
  return BTA_OK;
}
