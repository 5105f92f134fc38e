// Shared definitions for the botorch_amd HIP library (gfx950 / CDNA4).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>
#include <stddef.h>

#include "../../include/botorch_amd.h"

typedef double v4d __attribute__((ext_vector_type(4)));
typedef float v4f __attribute__((ext_vector_type(4)));
typedef double v2d __attribute__((ext_vector_type(2)));

namespace bta {

// Thread-local last-error text, returned by bta_last_error().
void set_error(const char* fmt, ...);
int hip_fail(hipError_t e, const char* what);
int num_cus();
double* pinned_host_buffer();  // 512 doubles, per thread; nullptr if unavailable

#define BTA_HIP(call)                                                   \
  do {                                                                  \
    hipError_t _e = (call);                                             \
    if (_e != hipSuccess) return ::bta::hip_fail(_e, #call);            \
  } while (0)

#define BTA_LAUNCH_CHECK(what)                                          \
  do {                                                                  \
    hipError_t _e = hipGetLastError();                                  \
    if (_e != hipSuccess) return ::bta::hip_fail(_e, what);             \
  } while (0)

inline int64_t round_up(int64_t x, int64_t m) { return (x + m - 1) / m * m; }

// Matern-5/2 / RBF value and the radial factor of its gradient, in scaled
// coordinates (x / lengthscale).  For r^2 = |xs - ts|^2:
//   Matern-5/2: k = s (1 + sqrt5 r + 5/3 r^2) exp(-sqrt5 r)
//               dk/dxs = -s 5/3 (1 + sqrt5 r) exp(-sqrt5 r) (xs - ts) = -h (xs - ts)
//   RBF:        k = s exp(-r^2/2),  dk/dxs = -s exp(-r^2/2) (xs - ts)
__device__ __forceinline__ double kern_value(int kind, double r2, double s) {
  if (kind == BTA_KERNEL_MATERN52) {
    double r = sqrt(r2);
    double sr = 2.2360679774997896964 * r;
    return s * (1.0 + sr + (5.0 / 3.0) * r2) * exp(-sr);
  }
  return s * exp(-0.5 * r2);
}

// returns h with dk/dxs = -h (xs - ts); also the value through *k
__device__ __forceinline__ double kern_grad_factor(int kind, double r2, double s, double* k) {
  if (kind == BTA_KERNEL_MATERN52) {
    double r = sqrt(r2);
    double sr = 2.2360679774997896964 * r;
    double e = exp(-sr);
    if (k) *k = s * (1.0 + sr + (5.0 / 3.0) * r2) * e;
    return s * (5.0 / 3.0) * (1.0 + sr) * e;
  }
  double e = exp(-0.5 * r2);
  if (k) *k = s * e;
  return s * e;
}

// e^x for x <= 0 (the kernels' arguments): Cody-Waite reduction x = k ln2 + f
// with ln2 split in two (|f| <= ln2/2), then the degree-12 Taylor polynomial
// of e^f (remainder < 2e-16 relative) and an exact power-of-two scaling.
// Below -745 the result underflows to 0; NaN propagates.
__host__ __device__ __forceinline__ double exp_nonpos(double x) {
  const bool under = x < -745.2;
  x = under ? 0.0 : x;
  const double kf = rint(x * 1.4426950408889634074);
  double f = fma(kf, -6.93147180369123816490e-01, x);
  f = fma(kf, -1.90821492927058770002e-10, f);
  double p = 1.0 / 479001600.0;  // 1/12!
  p = fma(p, f, 1.0 / 39916800.0);
  p = fma(p, f, 1.0 / 3628800.0);
  p = fma(p, f, 1.0 / 362880.0);
  p = fma(p, f, 1.0 / 40320.0);
  p = fma(p, f, 1.0 / 5040.0);
  p = fma(p, f, 1.0 / 720.0);
  p = fma(p, f, 1.0 / 120.0);
  p = fma(p, f, 1.0 / 24.0);
  p = fma(p, f, 1.0 / 6.0);
  p = fma(p, f, 0.5);
  p = fma(p, f, 1.0);
  p = fma(p, f, 1.0);
  return under ? 0.0 : ldexp(p, (int)kf);
}

// n / d for a normal d whose reciprocal is normal too: reciprocal seed, two Newton
// steps, and one residual correction of the quotient.
__host__ __device__ __forceinline__ double div_normal(double n, double d) {
#ifdef __HIP_DEVICE_COMPILE__
  double r = __builtin_amdgcn_rcp(d);
#else
  double r = (1.0 / d) * (1.0 + 0x1p-25);  // a seed as inexact as v_rcp_f64's
#endif
  r = fma(fma(-d, r, 1.0), r, r);
  r = fma(fma(-d, r, 1.0), r, r);
  const double q = n * r;
  return fma(fma(-d, q, n), r, q);
}

// log x for finite x > 0 (NaN gives NaN, infinity infinity; the callers hold x above 0):
// x = 2^k (1 + f) with 1 + f in [sqrt 1/2, sqrt 2), s = f / (2 + f), log(1 + f) =
// 2 atanh s summed as f - (f^2 / 2 - s (f^2 / 2 + R)) as in fdlibm, R = sum_{i >= 1}
// 2 s^2i / (2 i + 1) by its Taylor series to s^22 (remainder < 1e-18 relative), and
// k ln 2 in two parts.
__host__ __device__ __forceinline__ double log_pos(double x) {
  int k;
#ifdef __HIP_DEVICE_COMPILE__
  double m = __builtin_amdgcn_frexp_mant(x);
  k = __builtin_amdgcn_frexp_exp(x);
#else
  double m = frexp(x, &k);
#endif
  const bool low = m < 0.70710678118654752440;
  m = low ? m + m : m;
  const double kf = (double)(low ? k - 1 : k);
  const double f = m - 1.0;
  const double s = div_normal(f, 2.0 + f);
  const double z = s * s;
  double r = 2.0 / 23.0;
  r = fma(r, z, 2.0 / 21.0);
  r = fma(r, z, 2.0 / 19.0);
  r = fma(r, z, 2.0 / 17.0);
  r = fma(r, z, 2.0 / 15.0);
  r = fma(r, z, 2.0 / 13.0);
  r = fma(r, z, 2.0 / 11.0);
  r = fma(r, z, 2.0 / 9.0);
  r = fma(r, z, 2.0 / 7.0);
  r = fma(r, z, 2.0 / 5.0);
  r = fma(r, z, 2.0 / 3.0);
  r *= z;
  const double h = 0.5 * f * f;
  const double lo = fma(s, h + r, kf * 1.90821492927058770002e-10);
  const double v = fma(kf, 6.93147180369123816490e-01, f - (h - lo));
  return x <= 1.7976931348623157e308 ? v : x + x;
}

// sqrt(r2) for r2 >= 1e-30: v_rsq_f64 seed, one Goldschmidt step for the
// root and half-reciprocal pair, two Newton corrections of the root.
__device__ __forceinline__ double sqrt_pos(double r2) {
  const double y = __builtin_amdgcn_rsq(r2);
  double r = r2 * y, h = 0.5 * y;
  const double e = fma(-r, h, 0.5);
  r = fma(r, e, r);
  h = fma(h, e, h);
  double d = fma(-r, r, r2);
  r = fma(d, h, r);
  d = fma(-r, r, r2);
  return fma(d, h, r);
}

// Compile-time kernel kind: one code path per kernel instantiation.  The
// Matern distance is clamped at 1e-30 as gpytorch's MaternKernel does.
template <int KIND>
__device__ __forceinline__ double kern_value_k(double r2, double s) {
  if (KIND == BTA_KERNEL_MATERN52) {
    const double r = sqrt_pos(fmax(r2, 1e-30));
    const double sr = 2.2360679774997896964 * r;
    return s * (1.0 + sr + (5.0 / 3.0) * r2) * exp_nonpos(-sr);
  }
  return s * exp_nonpos(-0.5 * r2);
}

template <int KIND>
__device__ __forceinline__ double kern_grad_factor_k(double r2, double s) {
  if (KIND == BTA_KERNEL_MATERN52) {
    const double r = sqrt_pos(fmax(r2, 1e-30));
    const double sr = 2.2360679774997896964 * r;
    return s * (5.0 / 3.0) * (1.0 + sr) * exp_nonpos(-sr);
  }
  return s * exp_nonpos(-0.5 * r2);
}

// x / l with r = 1 / l (correctly rounded), equal to the division while x's residuals
// stay normal (|x| > 1e-290): q is within two ulps after the product, faithful after the
// first residual correction and correctly rounded after the second (Markstein,
// "Computation of elementary functions on the IBM RISC System/6000 processor", 1990).
// A product of 0 (also by an infinite l), infinity or NaN is the quotient already; its
// residual would be NaN or lose the sign.
__host__ __device__ __forceinline__ double div_by(double x, double l, double r) {
  const double q0 = x * r;
  const double q1 = fma(fma(-q0, l, x), r, q0);
  const double q2 = fma(fma(-q1, l, x), r, q1);
  return q0 != 0.0 && fabs(q0) < INFINITY ? q2 : q0;
}

// v of lane l of the wave (l uniform)
__device__ __forceinline__ double lane_bcast(double v, int l) {
  const int2 p = __builtin_bit_cast(int2, v);
  int2 r;
  r.x = __builtin_amdgcn_readlane(p.x, l);
  r.y = __builtin_amdgcn_readlane(p.y, l);
  return __builtin_bit_cast(double, r);
}

// v of lane (this lane ^ OFF), OFF = 1, 2, 4 or 8, by DPP moves within rows of 16
// lanes (every lane of the row active): no LDS traffic, where a shuffle is two
// ds_bpermute and their wait.
template <int CTRL>
__device__ __forceinline__ double dpp_d(double v) {
  const int2 p = __builtin_bit_cast(int2, v);
  int2 r;
  r.x = __builtin_amdgcn_update_dpp(0, p.x, CTRL, 0xF, 0xF, false);
  r.y = __builtin_amdgcn_update_dpp(0, p.y, CTRL, 0xF, 0xF, false);
  return __builtin_bit_cast(double, r);
}
template <int OFF>
__device__ __forceinline__ double row_xor(double v) {
  static_assert(OFF == 1 || OFF == 2 || OFF == 4 || OFF == 8, "within a row of 16");
  if constexpr (OFF == 1) return dpp_d<0xB1>(v);                // quad_perm [1, 0, 3, 2]
  else if constexpr (OFF == 2) return dpp_d<0x4E>(v);           // quad_perm [2, 3, 0, 1]
  else if constexpr (OFF == 4) return dpp_d<0x1B>(dpp_d<0x141>(v));  // i -> 7 - i -> i ^ 4
  else return dpp_d<0x128>(v);                                  // row_ror:8
}

// Exchanges the upper 32 lanes (OFF = 32) or the odd rows of 16 (OFF = 16) of a with
// the lower ones (the even rows) of b; all 64 lanes active.
template <int OFF>
__device__ __forceinline__ void lane_swap(double& a, double& b) {
  static_assert(OFF == 16 || OFF == 32, "half waves or rows");
#ifdef __HIP_DEVICE_COMPILE__
  uint2 x = __builtin_bit_cast(uint2, a), y = __builtin_bit_cast(uint2, b);
  if constexpr (OFF == 32) {
    const auto lo = __builtin_amdgcn_permlane32_swap(x.x, y.x, false, false);
    const auto hi = __builtin_amdgcn_permlane32_swap(x.y, y.y, false, false);
    x.x = lo[0], y.x = lo[1], x.y = hi[0], y.y = hi[1];
  } else {
    const auto lo = __builtin_amdgcn_permlane16_swap(x.x, y.x, false, false);
    const auto hi = __builtin_amdgcn_permlane16_swap(x.y, y.y, false, false);
    x.x = lo[0], y.x = lo[1], x.y = hi[0], y.y = hi[1];
  }
  a = __builtin_bit_cast(double, x);
  b = __builtin_bit_cast(double, y);
#endif
}

// op over the 64 lanes in the order of a butterfly of steps 32, 16, .., 1 (every lane
// gets the result).  The two first steps are one swap and one operation each: a step's
// two operands are the halves of the swapped copies.
template <typename OP>
__device__ __forceinline__ double wave_reduce(double v, OP op) {
  double w = v;
  lane_swap<32>(v, w);
  v = w = op(v, w);
  lane_swap<16>(v, w);
  v = op(v, w);
  v = op(v, row_xor<8>(v));
  v = op(v, row_xor<4>(v));
  v = op(v, row_xor<2>(v));
  return op(v, row_xor<1>(v));
}
__device__ __forceinline__ double wave_sum(double v) {
  return wave_reduce(v, [](double a, double b) { return a + b; });
}
__device__ __forceinline__ double wave_max(double v) {
  return wave_reduce(v, [](double a, double b) { return fmax(a, b); });
}
__device__ __forceinline__ double wave_min(double v) {
  return wave_reduce(v, [](double a, double b) { return fmin(a, b); });
}

// NV independent wave sums, each in the order of wave_sum.
template <int NV>
__device__ __forceinline__ void wave_sum_n(double (&v)[NV]) {
#pragma unroll
  for (int i = 0; i < NV; ++i) v[i] = wave_sum(v[i]);
}

// NV <= 32 wave sums with P - 1 + (6 - log2 P) exchanges instead of 6 NV
// (P = NV rounded up to a power of two): the first log2 P butterfly steps
// halve the values each lane carries (the lane with the step's bit set keeps
// the upper half, its partner the lower), the remaining steps are ordinary
// butterflies.  The total of value e ends in lanes e * 64/P .. (e + 1) * 64/P - 1;
// the first of them gets *e_out = e, every other lane -1 (also lanes past NV).
// Every value is summed over the same tree as wave_sum: bit-identical totals.
template <int OFF, int H, int P>
__device__ __forceinline__ void spread_step(double (&a)[P], int lane) {
  if constexpr (OFF >= 16) {  // a swap leaves both operands of every lane's sum
#pragma unroll
    for (int i = 0; i < H; ++i) {
      lane_swap<OFF>(a[i], a[H + i]);
      a[i] += a[H + i];
    }
  } else {
    const bool up = (lane & OFF) != 0;
#pragma unroll
    for (int i = 0; i < H; ++i) {
      // The empty asm (no instruction) makes lo and hi opaque values: without
      // it the compiler turns the lane-dependent choice below into a select of
      // the element index and extracts a[index] through compare/select chains
      // over the whole array (about 7x the instructions at NV = 10).
      double lo = a[i], hi = a[H + i];
      __asm__("" : "+v"(lo), "+v"(hi));
      const double keep = up ? hi : lo;
      const double send = up ? lo : hi;
      a[i] = keep + row_xor<OFF>(send);
    }
  }
}
template <int NV>
__device__ __forceinline__ double wave_sum_spread(const double (&v)[NV], int* e_out) {
  static_assert(NV >= 1 && NV <= 32, "wave_sum_spread: 1..32 values");
  constexpr int P = NV <= 1 ? 1 : NV <= 2 ? 2 : NV <= 4 ? 4 : NV <= 8 ? 8 : NV <= 16 ? 16 : 32;
  constexpr int LG = P == 1 ? 0 : P == 2 ? 1 : P == 4 ? 2 : P == 8 ? 3 : P == 16 ? 4 : 5;
  const int lane = threadIdx.x & 63;
  double a[P];
#pragma unroll
  for (int i = 0; i < P; ++i) a[i] = i < NV ? v[i] : 0.0;
  if constexpr (LG >= 1) spread_step<32, (P >> 1)>(a, lane);
  if constexpr (LG >= 2) spread_step<16, (P >> 2)>(a, lane);
  if constexpr (LG >= 3) spread_step<8, (P >> 3)>(a, lane);
  if constexpr (LG >= 4) spread_step<4, (P >> 4)>(a, lane);
  if constexpr (LG >= 5) spread_step<2, (P >> 5)>(a, lane);
  double t = a[0];
  if constexpr (LG == 0) {
    double w = t;
    lane_swap<32>(t, w);
    t += w;
  }
  if constexpr (LG <= 1) {
    double w = t;
    lane_swap<16>(t, w);
    t += w;
  }
  if constexpr (LG <= 2) t += row_xor<8>(t);
  if constexpr (LG <= 3) t += row_xor<4>(t);
  if constexpr (LG <= 4) t += row_xor<2>(t);
  t += row_xor<1>(t);
  const int e = lane >> (6 - LG);
  *e_out = ((lane & ((64 >> LG) - 1)) == 0 && e < NV) ? e : -1;
  return t;
}

}  // namespace bta
