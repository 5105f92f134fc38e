// Fused log-areas of qLogEHVI / qLogNEHVI: the reference's only native op
// (csrc/logei_fused.cpp:184-373, bound at acquisition/multi_objective/
// logei.py:107-170), as HIP kernels.
//
// For objective subsets obj[b][s][j][k] (b < B, s < n_sub subsets of size i,
// j < i, k < m objectives) and hyper-rectangle cells [cl, cu] (nc cells, shared
// or one set per b):
//   li[j][k]  = log_fatplus(obj[b][s][j][k] - cl[c][k], tau_relu)
//   lim[k]    = fatmin_j(li[j][k], tau_max)
//   lcl[k]    = log(min(cu[c][k], clamp) - cl[c][k])
//   out[b][c][s] = sum_k fatmin(lim[k], lcl[k], tau_max)
// (acquisition/multi_objective/logei.py:437-479, steps 1-4 of
// _compute_log_qehvi).  fatmin(x) = mn - tau log sum_j pareto((x_j - mn) / tau)
// with pareto(z) = 2 / (2 + 2z + z^2) and mn = the first minimum; its gradient
// goes to every x_j through the Pareto weights and to the first minimum through
// the 1 + ... term (csrc/logei_fused.cpp:117-177 has the same closed form).
//
// Forward: one thread per output element (b, c, s), the objective loop inside.
// Backward: the objectives do not mix, so (b, s, k) is independent; P neighbouring
// lanes share its cells (P a power of two up to 16, chosen so that the launch has a
// few waves per SIMD), accumulate d out / d obj[b][s][:][k] in registers (at most
// I_MAX = 32 subset members) and add up by shuffles in a fixed order.  Nothing is
// accumulated atomically.
//
// Both are bound by FP64 VALU work, so what they evaluate is trimmed: log(cell
// side) once per cell and block (LDS) instead of per element; the minimum's own
// Pareto term is exactly 1; the second fat minima's logs over the objectives are
// one log of the product of their sums (each in [1, 2]); exp is left out where it
// is below half an ulp of the Cauchy term beside it; logs by log_pos (about 35
// instructions against the math library's 90), divisions by div_normal.  4096 x 6
// pairs, 40 cells, 2 objectives: forward 49 -> 34 us, backward 95 (768 waves, one lane
// per (b, s, k)) -> 50 us; the call through autograd, which the host bounds, stays 126.
#include "bta_common.h"

namespace bta {

constexpr int LA_MAX_I = 32;
constexpr int LA_MAX_M = 8;
constexpr double LA_ALPHA = 0.1;  // Cauchy weight of the fat softplus

// Past these arguments exp(-|y|) is below half an ulp of what it is added to: 0.1 /
// (1 + y^2) in the value and 0.2 y / (1 + y^2)^2 in the derivative for y < 0, and 1
// in the sigmoid for y > 0.
constexpr double LA_FAR = 60.0;

template <typename T>
__device__ __forceinline__ T la_softplus(T y) {
  if (y > T(20)) return y;
  if (y < T(-LA_FAR)) return T(0);
  if (y < T(-20)) return exp(y);
  return log1p(exp(y));
}

template <typename T>
__device__ __forceinline__ T la_sigmoid(T y) {
  if (y > T(LA_FAR)) return T(1);
  if (y < T(-LA_FAR)) return T(0);
  if (y >= T(0)) return T(1) / (T(1) + exp(-y));
  const T e = exp(y);
  return e / (T(1) + e);
}

// n / d for 1 <= d; in FP64 0 where d is so large that its reciprocal would leave
// the normal range (div_normal would make NaN of an infinite d).
__device__ __forceinline__ double la_div(double n, double d) {
  return d < 1e307 ? div_normal(n, d) : (d >= 1e307 ? 0.0 : d);
}
__device__ __forceinline__ float la_div(float n, float d) { return n / d; }

// log of a positive argument (or NaN)
__device__ __forceinline__ double la_log(double x) { return log_pos(x); }
__device__ __forceinline__ float la_log(float x) { return log(x); }

// log(tau (softplus(x / tau) + 0.1 / (1 + (x / tau)^2))) and, when dv is not
// null, its derivative in x; a non-positive argument of the log gives -1e30.
template <typename T>
__device__ __forceinline__ T la_log_fatplus(T x, T tau, T inv_tau, T* dv) {
  const T y = x * inv_tau;
  const T cy = la_div(T(1), T(1) + y * y);
  const T f = la_softplus(y) + T(LA_ALPHA) * cy;
  const T tf = tau * f;
  if (!(tf > T(0))) {
    if (dv) *dv = T(0);
    return T(-1e30);
  }
  if (dv) *dv = (la_sigmoid(y) - T(2 * LA_ALPHA) * y * cy * cy) / tf;
  return la_log(tf);
}

// fatmin over x[0..n) = *mn_out - tau log S with S returned (1 where the fat
// minimum is the minimum itself); gw (n values) receives d fatmin / d x when
// want_grad.
template <typename T, int N>
__device__ __forceinline__ T la_fatmin(const T (&x)[N], int n, T inv_tau, T (&gw)[N],
                                       bool want_grad, T* mn_out) {
  T mn = x[0];
  int ami = 0;
#pragma unroll
  for (int j = 1; j < N; ++j)
    if (j < n && x[j] < mn) {
      mn = x[j];
      ami = j;
    }
  *mn_out = mn;
  if (n == 1 || mn < T(-1e29)) {
    if (want_grad)
#pragma unroll
      for (int j = 0; j < N; ++j) gw[j] = j == ami ? T(1) : T(0);
    return T(1);
  }
  // the minimum's own term: 1, with Pareto derivative -1
  T S = T(1), Sd = T(0);
#pragma unroll
  for (int j = 0; j < N; ++j) {
    if (j < n && j != ami) {
      const T z = (x[j] - mn) * inv_tau;
      const T den = T(2) + T(2) * z + z * z;
      const T p = la_div(T(2), den);
      S += p;
      if (want_grad) {
        gw[j] = -p * p * (T(1) + z);  // the Pareto derivative, turned into the weight below
        Sd += gw[j];
      }
    }
  }
  if (want_grad) {
    const T rS = la_div(T(1), S);
#pragma unroll
    for (int j = 0; j < N; ++j)
      if (j < n) gw[j] = j == ami ? T(1) + Sd * rS : -gw[j] * rS;
  }
  return S;
}

template <typename T>
struct LaArgs {
  const T* obj;  // B x n_sub x i x m
  const T* cl;   // B_cells x nc x m
  const T* cu;
  const T* g_out;  // B x nc x n_sub (backward)
  T* out;          // forward: B x nc x n_sub; backward: B x n_sub x i x m
  int64_t B, n_sub, B_cells, nc;
  int i, m;
  T tau_relu, tau_max, clamp;
};

// log of the cell sides, nc x m, for a block's threads (lcl in LDS); TAB is chosen
// when every batch element has the same cells and they fit
constexpr int LA_TAB = 1024;

template <typename T>
__device__ __forceinline__ T la_log_side(const LaArgs<T>& a, int64_t i) {
  return log(fmin(a.cu[i], a.clamp) - a.cl[i]);
}

template <typename T, bool TAB>
__device__ __forceinline__ void la_fill_sides(const LaArgs<T>& a, T* lcl) {
  if (!TAB) return;
  for (int i = threadIdx.x; i < (int)a.nc * a.m; i += 256) lcl[i] = la_log_side(a, i);
  __syncthreads();
}

template <typename T, int I, bool TAB>
__global__ __launch_bounds__(256) void log_areas_fwd_kernel(LaArgs<T> a) {
  __shared__ T lcl[TAB ? LA_TAB : 1];
  la_fill_sides<T, TAB>(a, lcl);
  const int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int64_t total = a.B * a.nc * a.n_sub;
  if (e >= total) return;
  const int64_t s = e % a.n_sub, c = (e / a.n_sub) % a.nc, b = e / (a.n_sub * a.nc);
  const int64_t bc = a.B_cells == 1 ? 0 : b;
  const T* o = a.obj + (b * a.n_sub + s) * a.i * a.m;
  const int64_t cell = (bc * a.nc + c) * a.m;
  const T itr = T(1) / a.tau_relu, itm = T(1) / a.tau_max;
  T area = T(0), S = T(1);
  for (int k = 0; k < a.m; ++k) {
    const T lk = a.cl[cell + k];
    T li[I], unused[I], mn;
#pragma unroll
    for (int j = 0; j < I; ++j)
      li[j] = j < a.i ? la_log_fatplus<T>(o[j * a.m + k] - lk, a.tau_relu, itr, nullptr) : T(0);
    const T s1 = la_fatmin<T, I>(li, a.i, itm, unused, false, &mn);
    if (a.i > 1) mn -= a.tau_max * la_log(s1);
    T pair[2] = {mn, TAB ? lcl[cell + k] : la_log_side(a, cell + k)};
    T g2[2];
    S *= la_fatmin<T, 2>(pair, 2, itm, g2, false, &mn);
    area += mn;
  }
  a.out[e] = area - a.tau_max * la_log(S);
}

template <typename T, int I, bool TAB>
__global__ __launch_bounds__(256) void log_areas_bwd_kernel(LaArgs<T> a, int P) {
  __shared__ T lcl[TAB ? LA_TAB : 1];
  la_fill_sides<T, TAB>(a, lcl);
  const int64_t gid = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int64_t e = gid / P;  // (P divides the wave: its lanes stay together)
  const int part = (int)(gid % P);
  const int64_t total = a.B * a.n_sub * a.m;
  if (e >= total) return;
  const int k = (int)(e % a.m);
  const int64_t s = (e / a.m) % a.n_sub, b = e / (a.m * a.n_sub);
  const int64_t bc = a.B_cells == 1 ? 0 : b;
  const T* o = a.obj + (b * a.n_sub + s) * a.i * a.m;
  const T itr = T(1) / a.tau_relu, itm = T(1) / a.tau_max;
  T ok[I], g[I];
#pragma unroll
  for (int j = 0; j < I; ++j) {
    ok[j] = j < a.i ? o[j * a.m + k] : T(0);
    g[j] = T(0);
  }
  for (int64_t c = part; c < a.nc; c += P) {
    const int64_t cell = (bc * a.nc + c) * a.m + k;
    const T lk = a.cl[cell];
    const T go = a.g_out[(b * a.nc + c) * a.n_sub + s];
    T li[I], lg[I], fw[I], mn;
#pragma unroll
    for (int j = 0; j < I; ++j) {
      T d = T(0);
      li[j] = j < a.i ? la_log_fatplus<T>(ok[j] - lk, a.tau_relu, itr, &d) : T(0);
      lg[j] = d;
    }
    const T s1 = la_fatmin<T, I>(li, a.i, itm, fw, true, &mn);
    if (a.i > 1) mn -= a.tau_max * la_log(s1);
    T pair[2] = {mn, TAB ? lcl[cell] : la_log_side(a, cell)};
    T g2[2];
    la_fatmin<T, 2>(pair, 2, itm, g2, true, &mn);
    const T gl = go * g2[0];
#pragma unroll
    for (int j = 0; j < I; ++j)
      if (j < a.i) g[j] += gl * fw[j] * lg[j];
  }
  T* go = a.out + (b * a.n_sub + s) * a.i * a.m;
#pragma unroll
  for (int j = 0; j < I; ++j) {
    if (j >= a.i) break;
    T v = g[j];
    for (int off = P / 2; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
    if (part == 0) go[j * a.m + k] = v;
  }
}

template <typename T>
static int log_areas_launch(bool bwd, const LaArgs<T>& a, hipStream_t st) {
  const int64_t items = bwd ? a.B * a.n_sub * a.m : a.B * a.nc * a.n_sub;
  if (items == 0) return BTA_OK;
  // backward: lanes per item until the launch has about eight waves per SIMD
  int P = 1;
  if (bwd)
    while (P < 16 && 2 * P <= a.nc && items * P < (int64_t)num_cus() * 4 * 8 * 64) P *= 2;
  const dim3 grid((unsigned)((items * P + 255) / 256));
  const int I = a.i <= 4 ? 4 : a.i <= 8 ? 8 : a.i <= 16 ? 16 : 32;
  const bool tab = a.B_cells == 1 && a.nc <= 256 && a.nc * a.m <= LA_TAB;
#define LA_GO2(II, TT)                                                                        \
  if (bwd) hipLaunchKernelGGL((log_areas_bwd_kernel<T, II, TT>), grid, dim3(256), 0, st, a, P); \
  else hipLaunchKernelGGL((log_areas_fwd_kernel<T, II, TT>), grid, dim3(256), 0, st, a);
#define LA_GO(II)              \
  if (tab) { LA_GO2(II, true) } \
  else { LA_GO2(II, false) }
  switch (I) {
    case 4: LA_GO(4) break;
    case 8: LA_GO(8) break;
    case 16: LA_GO(16) break;
    default: LA_GO(32) break;
  }
#undef LA_GO
#undef LA_GO2
  BTA_LAUNCH_CHECK(bwd ? "log_areas_bwd_kernel" : "log_areas_fwd_kernel");
  return BTA_OK;
}

static int log_areas(bool bwd, int f32, const void* g_out, const void* obj, int64_t B,
                     int64_t n_sub, int i, int m, const void* cl, const void* cu, int64_t B_cells,
                     int64_t nc, double tau_relu, double tau_max, void* out, hipStream_t st) {
  if (!obj || !cl || !cu || !out || (bwd && !g_out) || B < 0 || n_sub < 0 || nc < 0 ||
      i < 1 || i > LA_MAX_I || m < 1 || m > LA_MAX_M || !(B_cells == 1 || B_cells == B) ||
      !(tau_relu > 0.0) || !(tau_max > 0.0) || B * nc * n_sub > ((int64_t)1 << 40)) {
    set_error("log_areas: invalid arguments (need 1 <= i <= %d, 1 <= m <= %d, B_cells 1 or B, "
              "positive temperatures)",
              LA_MAX_I, LA_MAX_M);
    return BTA_ERR_INVALID;
  }
  if (f32) {
    LaArgs<float> a{(const float*)obj, (const float*)cl, (const float*)cu, (const float*)g_out,
                    (float*)out, B, n_sub, B_cells, nc, i, m, (float)tau_relu,
                    (float)tau_max, 1e8f};
    return log_areas_launch<float>(bwd, a, st);
  }
  LaArgs<double> a{(const double*)obj, (const double*)cl, (const double*)cu,
                   (const double*)g_out, (double*)out, B, n_sub, B_cells, nc, i, m, tau_relu,
                   tau_max, 1e10};
  return log_areas_launch<double>(bwd, a, st);
}

}  // namespace bta

extern "C" int bta_log_areas_forward(int32_t f32, const void* obj, int64_t B, int64_t n_sub,
                                     int32_t i, int32_t m, const void* cell_lower,
                                     const void* cell_upper, int64_t B_cells, int64_t nc,
                                     double tau_relu, double tau_max, void* out,
                                     bta_stream_t stream) {
  return bta::log_areas(false, f32, nullptr, obj, B, n_sub, i, m, cell_lower, cell_upper,
                        B_cells, nc, tau_relu, tau_max, out, (hipStream_t)stream);
}

extern "C" int bta_log_areas_backward(int32_t f32, const void* grad_out, const void* obj,
                                      int64_t B, int64_t n_sub, int32_t i, int32_t m,
                                      const void* cell_lower, const void* cell_upper,
                                      int64_t B_cells, int64_t nc, double tau_relu,
                                      double tau_max, void* grad_obj, bta_stream_t stream) {
  return bta::log_areas(true, f32, grad_out, obj, B, n_sub, i, m, cell_lower, cell_upper,
                        B_cells, nc, tau_relu, tau_max, grad_obj, (hipStream_t)stream);
}
