// The per-restart MC stage of the qLogNEI step and its adjoint (mc_body), the
// per-model launch arguments of the whole step (StepArgs), shared by the
// one-model step (qlognei.hip) and the step over many models (qbatch.hip).
// The algorithm is described at the top of qlognei.hip.
#pragma once
#include <cstdlib>

#include "bta_common.h"
#include "gemm.h"
#include "gemm_h2_body.h"
#include "kernels.h"

namespace bta {

constexpr int MC_MAXD = 32;
constexpr int MC_MAXNB_SLOTS = 4;  // n_b <= 256
constexpr int MC_LB_STAGE = 16;    // Lb staged in LDS for n_b up to this
// LDS bound of the MC stage, the same for the standalone and the fused
// launches so that a state is accepted by both or by neither (the value-only
// call runs the standalone kernel, value+grad may run the fused one).
constexpr size_t MC_LDS_MAX = 64 * 1024;

struct McArgs {
  const void* vt;
  int64_t ldv;
  double* gq;         // R x q: dV = gq V per restart block (-2 s^2 gA)
  const double* xs;
  const double* bs;
  const double* Lb;
  const double* Lb_levels;  // joint mode: chol(Sigma_bb + j_t I), t = 0..max_tries, or NULL
  int lb_levels_mask;       // bit t: Lb_levels[t] exists
  const double* Zt;
  const double* best_f;
  const double* P;    // R x ne x p_parts partial sums of K_x [alpha | A] (FP64)
  int p_parts;
  double* dext;       // R x ne: adjoint of P
  double* value;
  double* dxs_extra;
  int* status;
  int d, n_pad, n_b, S, kind, max_tries, grad;
  int nrest;  // restarts (b)
  int nr;     // restarts per MC workgroup (1 or 2; mc_paired)
  double outputscale, y_mean, y_std, c, tau_relu, tau_max, jitter;
};

// LDS layout (doubles) shared by host sizing and the kernel.
struct McLayout {
  int xq, red, mu, dmu, sqq, lbr, ga, lnew, dlnew, dsqb, u, G, scal, pv, vv, hh, lb, lb_n, total;
  __host__ __device__ McLayout(int Q, int n_b, int S) {
    const int m = n_b + Q;
    int o = 0;
    xq = o; o += Q * MC_MAXD;
    red = o; o += 4 * 64;
    pv = o; o += Q * (n_b + 1);
    vv = o; o += Q * (Q + 1) / 2;
    hh = o; o += Q * m;
    mu = o; o += Q;
    dmu = o; o += Q;
    sqq = o; o += Q * Q;
    lbr = o; o += Q * Q;
    ga = o; o += Q * Q;
    lnew = o; o += Q * m;
    dlnew = o; o += Q * m;
    dsqb = o; o += Q * (n_b > 0 ? n_b : 1);
    u = o; o += S;
    G = o; o += S * Q;
    scal = o; o += 8;
    // Lb (n_b x n_b) for the triangular solves, when n_b <= MC_LB_STAGE and it
    // keeps the layout within MC_LDS_MAX
    lb = o;
    lb_n = n_b <= MC_LB_STAGE && (size_t)(o + n_b * n_b) * sizeof(double) <= MC_LDS_MAX
               ? n_b * n_b : 0;
    o += lb_n;
    total = o;
  }
};

// Two restarts per MC workgroup (two waves each) in the split-FP16 mixed mode
// with q <= 5, whose MC workgroups share the CUs with the adjoint GEMM's
// workers in one launch (one round of paired workgroups in the slots the
// workers leave free is shorter than two rounds of single ones), when both
// layouts fit MC_LDS_MAX and the cached root is in use (not the joint mode).
// Every launch of that mode's MC stage (fused or alone, value-only or with the
// gradient, one model or many) takes the same choice, kept in McArgs::nr when
// the step's arguments are built, and a restart's results depend only on it,
// not on the partner restart, so value-only and value+grad steps, chunked or
// whole, one model or many, keep giving identical values.  Run alone over the
// whole GPU (mixed_f32), single workgroups fill both slots of every CU and
// stay.  BTA_MC_PAIR=0 in the environment keeps one restart per workgroup (how
// the two are compared in the tests).
inline bool mc_paired(const McArgs& a, int q, bool f32, bool split) {
  const char* e = getenv("BTA_MC_PAIR");
  const McLayout lay(q, a.n_b, a.S);
  return f32 && split && q <= 5 && !a.Lb_levels && !(e && e[0] == '0') &&
         (size_t)2 * lay.total * sizeof(double) <= MC_LDS_MAX;
}

// a / b in TM: FP32 takes the hardware reciprocal (1 ulp) and a product, FP64
// divides exactly
template <typename TM>
__device__ __forceinline__ TM div_tm(TM a, TM b) {
  if constexpr (sizeof(TM) == 4) return a * __builtin_amdgcn_rcpf(b);
  else return a / b;
}

// log(tau * (softplus(x/tau) + 0.1 / (1 + (x/tau)^2))) and its derivative
// (utils/safe_math.py:298-325), evaluated in TM (FP64, or FP32 for the mixed
// modes' sample arithmetic) from the FP64 difference x; rtau = 1 / tau.
//
// In FP32, log1p(e) follows Goldberg's rule log(u) e / (u - 1), u = 1 + e (a few
// ulp; "What every computer scientist should know about floating-point
// arithmetic", 1991, thm. 4), and the divisions use div_tm.
//
// In FP64 log1p(e) = log u + (e - (u - 1)) / u, whose correction is at most an ulp of
// u, so the hardware reciprocal is enough for it; logs, exponentials and quotients
// are those of bta_common.h, without the general forms' branches for operands that
// cannot occur (z^2 and its products are held below 1e300 so that every divisor and
// its reciprocal stay normal).  With the library's forms and exact divisions the
// samples of one candidate took 9400 cycles of a 49900-cycle workgroup, now 7200 of 32000.
template <typename TM>
__device__ __forceinline__ void log_fatplus_grad(double x, double tau, double rtau, double* v,
                                                 double* dv) {
  constexpr bool f32 = sizeof(TM) == 4;
  const TM z = (TM)(x * rtau);
  TM sp, sig;
  if constexpr (f32) {
    if (z > (TM)20) {  // torch softplus threshold
      sp = z;
      sig = (TM)1;
    } else {
      const TM e = exp(z);
      const TM u = (TM)1 + e;
      sp = u == (TM)1 ? e : log(u) * div_tm(e, u - (TM)1);
      sig = div_tm(e, u);
    }
    const TM z2 = (TM)1 + z * z;
    const TM cz = div_tm((TM)1, z2);
    const TM f = sp + (TM)0.1 * cz;
    const TM tt = (TM)tau;
    *v = (double)log(tt * f);
    // dv = (sig - 0.2 z cz^2) / (f tau), with cz / f = 1 / (sp (1 + z^2) + 0.1) so
    // that no intermediate underflows for large |z|
    const TM cf = sp > (TM)0 ? div_tm((TM)1, sp * z2 + (TM)0.1) : (TM)10;
    const TM g = div_tm(sig, f) - (TM)0.2 * z * cz * cf;
    *dv = (double)(g * (TM)rtau);
  } else {
    const bool lin = z > 20.0;
    const double e = exp_nonpos(lin ? 0.0 : z);  // (its reduction holds up to e^20)
    const double u = 1.0 + e;
    const double l1p = fma(e - (u - 1.0), __builtin_amdgcn_rcp(u), log_pos(u));
    sp = lin ? z : l1p;
    sig = lin ? 1.0 : div_normal(e, u);
    double z2 = fma(z, z, 1.0);
    z2 = z2 > 1e300 ? 1e300 : z2;
    const double cz = div_normal(1.0, z2);
    const double f = fma(0.1, cz, sp);
    *v = log_pos(tau * f);
    double t = fma(sp, z2, 0.1);
    t = t > 1e300 ? 1e300 : t;
    const double cf = div_normal(1.0, t);
    const double g = div_normal(sig, f) - 0.2 * z * cz * cf;
    *dv = g * rtau;
  }
}

// Triangular solves with the baseline factor L (n_b x n_b, row-major) for the Q rows of
// x (pitch px): x <- x L^-T (forward) or out <- x L^-1 (back), the subtractions of an
// element in column order.  Columns are eliminated one after the other, so the chain
// per column counts: a quotient by the reciprocal of the diagonal (div_by), a broadcast
// by DPP or readlane and one product.  Coefficients outside the triangle are zero, so a
// finished element stays as it is, still to be divided at the end: no lane masks on the
// chain.  (With an exact division, a shuffle and an LDS read per column a solve of 8
// columns took 8100 cycles, now 2600.)  EXACT: quotients equal to the division's; else
// (the FP64 mode) x times the reciprocal, six operations fewer on the chain.
//
// Up to 16 columns: four rows per wave, lane 16 r + j holding column j of row r and its
// coefficients in registers.
template <bool EXACT>
__device__ __forceinline__ double solve_quot(double x, double ld, double rd) {
  return EXACT ? div_by(x, ld, rd) : x * rd;
}
template <int U, bool EXACT>
__device__ __forceinline__ void solve16_step(double& x, const double (&c)[16], double ld,
                                             double rd) {
  // (0x150 + U: row_newbcast, lane U of each row of 16)
  x = fma(-c[U], dpp_d<0x150 | U>(solve_quot<EXACT>(x, ld, rd)), x);
}
template <int G, bool BACK, bool EXACT>
__device__ __forceinline__ void solve16_four(double& x, const double (&c)[16], double ld,
                                             double rd) {
  solve16_step<4 * G + (BACK ? 3 : 0), EXACT>(x, c, ld, rd);
  solve16_step<4 * G + (BACK ? 2 : 1), EXACT>(x, c, ld, rd);
  solve16_step<4 * G + (BACK ? 1 : 2), EXACT>(x, c, ld, rd);
  solve16_step<4 * G + (BACK ? 0 : 3), EXACT>(x, c, ld, rd);
}
template <int Q, bool BACK, bool EXACT>
__device__ __forceinline__ void solve16(const double* L, int n_b, const double* x, int px,
                                        double* out, int po, int wv, int wpr) {
  const int lane = threadIdx.x & 63, j = min(lane & 15, n_b - 1);
  const double ld = L[j * n_b + j], rd = 1.0 / ld;
  double c[16];
#pragma unroll
  for (int u = 0; u < 16; ++u) {
    const int k = min(u, n_b - 1);
    const double l = BACK ? L[k * n_b + j] : L[j * n_b + k];
    c[u] = (BACK ? j < u && u < n_b : j > u) ? l : 0.0;
  }
  for (int i0 = 4 * wv; i0 < Q; i0 += 4 * wpr) {  // (uniform over the wave)
    const int i = min(i0 + (lane >> 4), Q - 1);
    double v = x[i * px + j];
    if constexpr (BACK) {
      if (n_b > 12) solve16_four<3, true, EXACT>(v, c, ld, rd);
      if (n_b > 8) solve16_four<2, true, EXACT>(v, c, ld, rd);
      if (n_b > 4) solve16_four<1, true, EXACT>(v, c, ld, rd);
      solve16_four<0, true, EXACT>(v, c, ld, rd);
    } else {
      solve16_four<0, false, EXACT>(v, c, ld, rd);
      if (n_b > 4) solve16_four<1, false, EXACT>(v, c, ld, rd);
      if (n_b > 8) solve16_four<2, false, EXACT>(v, c, ld, rd);
      if (n_b > 12) solve16_four<3, false, EXACT>(v, c, ld, rd);
    }
    v = solve_quot<EXACT>(v, ld, rd);
    if ((lane & 15) < n_b && i0 + (lane >> 4) < Q) out[i * po + j] = v;
  }
}
// Any n_b (up to 256): one wave per row, lane l holding columns l + 64 t; 16 columns
// are eliminated within their slot, then taken off the other slots.  (Lanes past n_b
// repeat the last column and store nothing.)
template <int Q, bool BACK, bool EXACT>
__device__ __forceinline__ void solve_any(const double* L, int n_b, const double* x, int px,
                                          double* out, int po, int wv, int wpr) {
  constexpr int NS = MC_MAXNB_SLOTS;
  const int lane = threadIdx.x & 63;
  const int nc = (n_b + 15) / 16;
  for (int i = wv; i < Q; i += wpr) {
    double v[NS], ld[NS], rd[NS];
#pragma unroll
    for (int t = 0; t < NS; ++t) {
      const int j = min(lane + 64 * t, n_b - 1);
      v[t] = x[i * px + j];
      ld[t] = L[j * n_b + j];
    }
#pragma unroll
    for (int t = 0; t < NS; ++t) rd[t] = 1.0 / ld[t];
    for (int ci = 0; ci < nc; ++ci) {
      const int k0 = 16 * (BACK ? nc - 1 - ci : ci), ks = k0 >> 6;
      double y[16];
#pragma unroll
      for (int t0 = 0; t0 < NS; ++t0) {
        // the chunk's own slot first, then the others that still depend on it
        const int t = BACK ? NS - 1 - t0 : t0;
        if ((BACK ? t > ks : t < ks) || 64 * t >= n_b) continue;
        const int j = lane + 64 * t, jc = min(j, n_b - 1);
        double c[16];
#pragma unroll
        for (int u = 0; u < 16; ++u) {
          const int k = k0 + u, kc = min(k, n_b - 1);
          const double l = BACK ? L[kc * n_b + jc] : L[jc * n_b + kc];
          c[u] = (BACK ? j < k && k < n_b : j > k) ? l : 0.0;
        }
        if (t == ks) {
#pragma unroll
          for (int u0 = 0; u0 < 16; ++u0) {
            const int u = BACK ? 15 - u0 : u0;
            y[u] = lane_bcast(solve_quot<EXACT>(v[t], ld[t], rd[t]), (k0 + u) & 63);
            v[t] = fma(-c[u], y[u], v[t]);
          }
        } else {
#pragma unroll
          for (int u0 = 0; u0 < 16; ++u0) {
            const int u = BACK ? 15 - u0 : u0;
            v[t] = fma(-c[u], y[u], v[t]);
          }
        }
      }
    }
#pragma unroll
    for (int t = 0; t < NS; ++t) {
      const int j = lane + 64 * t;
      const double q = solve_quot<EXACT>(v[t], ld[t], rd[t]);
      if (j < n_b) out[i * po + j] = q;
    }
  }
}

// Reductions over the WPR waves of one restart (wave w of the restart writes
// red[w * 64 ...]); every thread of the restart gets the result.  The sums
// take the waves in order, after a fixed-tree sum within each wave.  Every
// thread of the workgroup must call them (they hold workgroup barriers).
template <int NV, int WPR>
__device__ __forceinline__ void group_sum(double (&v)[NV], double* red, double (&out)[NV], int wv) {
  if (NV <= 32) {
    int e;
    const double s =
        wave_sum_spread<(NV <= 32 ? NV : 1)>(*(const double(*)[NV <= 32 ? NV : 1])v, &e);
    if (e >= 0) red[wv * 64 + e] = s;
  } else {
    double s[NV];
#pragma unroll
    for (int i = 0; i < NV; ++i) s[i] = v[i];
    wave_sum_n<NV>(s);
    if ((threadIdx.x & 63) == 0)
#pragma unroll
      for (int i = 0; i < NV; ++i) red[wv * 64 + i] = s[i];
  }
  __syncthreads();
#pragma unroll
  for (int i = 0; i < NV; ++i) {
    double t = red[i];
#pragma unroll
    for (int w = 1; w < WPR; ++w) t += red[w * 64 + i];
    out[i] = t;
  }
  __syncthreads();
}

template <int WPR>
__device__ __forceinline__ double group_max1(double v, double* red, int wv) {
  const double s = wave_max(v);
  if ((threadIdx.x & 63) == 0) red[wv * 64] = s;
  __syncthreads();
  double r = red[0];
#pragma unroll
  for (int w = 1; w < WPR; ++w) r = fmax(r, red[w * 64]);
  __syncthreads();
  return r;
}

// |a - b|^2, eight coordinates loaded at a time
__device__ __forceinline__ double sq_dist(const double* a, const double* b, int d) {
  double r2 = 0.0;
  for (int j0 = 0; j0 < d; j0 += 8) {
    double x[8], y[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      const int j = min(j0 + u, d - 1);
      x[u] = a[j];
      y[u] = b[j];
    }
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      const double df = x[u] - y[u];
      if (j0 + u < d) r2 = fma(df, df, r2);
    }
  }
  return r2;
}

// Cholesky of a Q x Q matrix by one wave, lane i holding row i (lanes past Q repeat the
// last): ar its row of the matrix, l its row of the factor (entries right of the
// diagonal are not meaningful).  False at a pivot that is not positive.
template <int Q>
__device__ __forceinline__ bool small_chol(const double (&ar)[Q], double jit, int i,
                                           double (&l)[Q]) {
#pragma unroll
  for (int j = 0; j < Q; ++j) {
    double t = i == j ? ar[j] + jit : ar[j];
#pragma unroll
    for (int k = 0; k < j; ++k) t = fma(-l[k], lane_bcast(l[k], j), t);
    const double s = lane_bcast(t, j);
    if (!(s > 0.0)) return false;
    const double dj = sqrt(s), rdj = 1.0 / dj;
    l[j] = i == j ? dj : t * rdj;
  }
  return true;
}

// The MC stage and its adjoint for NR restarts per workgroup (NR = 1 or 2):
// restart bw * NR + h runs on threads [h TPR, (h + 1) TPR) with the McLayout
// area sm_all + h * total in LDS.  With NR = 2 the two restarts pass the same
// barriers, so their serial phases overlap; a half past the last restart
// repeats the last one and stores nothing.
template <int Q, typename TV, int NR = 1>
__device__ __forceinline__ void mc_body(const McArgs& a, const int bw, double* sm_all) {
  static_assert(NR == 1 || NR == 2, "one or two restarts per workgroup");
  constexpr int TPR = 256 / NR, WPR = 4 / NR;  // threads and waves per restart
  const McLayout lay(Q, a.n_b, a.S);
  const int half = (int)threadIdx.x / TPR;
  const int tid = (int)threadIdx.x % TPR, lane = tid & 63, wv = tid >> 6;
  const int bt = bw * NR + half;
  const bool live = bt < a.nrest;
  const int b = live ? bt : a.nrest - 1;
  double* sm = sm_all + half * lay.total;
  const int d = a.d, n_b = a.n_b, S = a.S, m = n_b + Q;
  const double ys = a.y_std, ys2 = a.y_std * a.y_std;
  double* xq = sm + lay.xq;
  double* red = sm + lay.red;
  double* mu = sm + lay.mu;
  double* dmu = sm + lay.dmu;
  double* sqq = sm + lay.sqq;
  double* lbr = sm + lay.lbr;
  double* gA = sm + lay.ga;
  double* lnew = sm + lay.lnew;
  double* dlnew = sm + lay.dlnew;
  double* dsqb = sm + lay.dsqb;
  double* uu = sm + lay.u;
  double* G = sm + lay.G;
  double* scal = sm + lay.scal;
  const TV* vt = (const TV*)a.vt;
  const int64_t r0 = (int64_t)b * Q;

  // the query coordinates (the first TPR one per thread, the rest, for q d >
  // TPR, after), then the restart's V rows for V_b V_b^T (16-byte loads): their
  // first two column passes are issued here, ahead of the other loads of the
  // stage
  const bool has_x = tid < Q * d;
  const double xr = has_x ? a.xs[r0 * d + tid] : 0.0;
  constexpr int VW = 16 / (int)sizeof(TV);  // elements per 16-byte load
  typedef TV vec_t __attribute__((ext_vector_type(VW)));
  vec_t vpre[2][Q];
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    const int k = (tid + TPR * h) * VW;
#pragma unroll
    for (int i = 0; i < Q; ++i)
      vpre[h][i] = k < a.n_pad ? *(const vec_t*)(vt + (r0 + i) * a.ldv + k) : vec_t{};
  }
  // In the cached-root mode Lb goes to LDS (lay.lb_n entries) for the two
  // triangular solves, whose column loops would otherwise wait on a global load
  // per step; the first TPR entries load here, with the V rows.
  const bool joint = a.Lb_levels != nullptr;
  const bool lb_lds = !joint && lay.lb_n > 0;
  double* lbs = sm + lay.lb;
  const double lbv = lb_lds && tid < lay.lb_n ? a.Lb[tid] : 0.0;
  if (has_x) xq[(tid / d) * MC_MAXD + tid % d] = xr;
  for (int i = tid + TPR; i < Q * d; i += TPR) xq[(i / d) * MC_MAXD + i % d] = a.xs[r0 * d + i];
  if (tid == 0) scal[1] = 0.0;
  __syncthreads();
  // Kernel values K(x_i, x_j) into sqq and K(x_i, X_b) into lnew[:, :n_b], and
  // with the gradient the radial factors of the direct input gradient into hh
  // (Q x m: h(x_i, x_j) for j < Q, 0 on the diagonal, h(x_i, b_kb) after); they
  // need only the coordinates, so they run (from the last wave down) while the
  // V rows and the P partials are in flight.
  double* hh = sm + lay.hh;
  for (int t = TPR - 1 - tid; t < Q * Q + Q * n_b; t += TPR) {
    if (t < Q * Q) {
      const int i = t / Q, j = t % Q;
      const double r2 = sq_dist(xq + i * MC_MAXD, xq + j * MC_MAXD, d);
      sqq[t] = kern_value(a.kind, r2, a.outputscale);
      if (a.grad)
        hh[i * m + j] = j == i ? 0.0 : kern_grad_factor(a.kind, r2, a.outputscale, nullptr);
    } else {
      const int e = t - Q * Q, i = e / n_b, kb = e % n_b;
      const double r2 = sq_dist(xq + i * MC_MAXD, a.bs + kb * d, d);
      lnew[i * m + kb] = kern_value(a.kind, r2, a.outputscale);
      if (a.grad) hh[i * m + Q + kb] = kern_grad_factor(a.kind, r2, a.outputscale, nullptr);
    }
  }

  // ---- P rows (fixed-order sums of their column-tile partials, one value per
  // wave task, partials across the lanes) and V_b V_b^T over the n_pad
  // columns of V (16-byte loads, all issued before the products) ----------
  constexpr int NQ = Q * (Q + 1) / 2;
  double* pv = sm + lay.pv;  // Q x (n_b + 1): P[r0 + i][j]
  double* vv = sm + lay.vv;  // packed lower triangle of V_b V_b^T
  constexpr bool ZPRE = Q <= 4;  // (the registers of more rows are taken)
  double zpre[2][8], bpre[2];
  {
    // 16 tasks per wave per pass, their loads issued together; each task's sum is
    // the same whatever the batch
    constexpr int TB = 16;
    const int ne = n_b + 1;
    for (int t0 = wv * TB; t0 < Q * ne; t0 += TB * WPR) {
      double s[TB];
#pragma unroll
      for (int u = 0; u < TB; ++u) s[u] = 0.0;
      const double* p = a.P + (r0 * ne + t0) * a.p_parts;
      const int last = Q * ne - 1 - t0;
      for (int pt = lane; pt < a.p_parts; pt += 64) {
        double x[TB];
#pragma unroll
        for (int u = 0; u < TB; ++u) x[u] = p[(int64_t)min(u, last) * a.p_parts + pt];
#pragma unroll
        for (int u = 0; u < TB; ++u) s[u] += x[u];
      }
      int e;
      const double tot = wave_sum_spread<TB>(s, &e);
      if (e >= 0 && t0 + e < Q * ne) pv[t0 + e] = tot;
    }
    double acc[NQ];
#pragma unroll
    for (int i = 0; i < NQ; ++i) acc[i] = 0.0;
    auto vv_pass = [&](const vec_t(&v)[Q]) {
#pragma unroll
      for (int e = 0; e < VW; ++e) {
        int idx = 0;
#pragma unroll
        for (int i = 0; i < Q; ++i)
#pragma unroll
          for (int j = 0; j <= i; ++j) {
            acc[idx] = fma((double)v[i][e], (double)v[j][e], acc[idx]);
            ++idx;
          }
      }
    };
#pragma unroll
    for (int h = 0; h < 2; ++h)
      if ((tid + TPR * h) * VW < a.n_pad) vv_pass(vpre[h]);
    for (int k = (tid + 2 * TPR) * VW; k < a.n_pad; k += TPR * VW) {
      vec_t v[Q];
#pragma unroll
      for (int i = 0; i < Q; ++i) v[i] = *(const vec_t*)(vt + (r0 + i) * a.ldv + k);
      vv_pass(v);
    }
    // the first eight base samples of this thread's first two samples, for the sample
    // stage: they arrive during the reductions and the solves
    if (ZPRE) {
      const int s0 = min(tid, S - 1), s1 = tid + TPR < S ? tid + TPR : s0;
      bpre[0] = a.best_f[s0];
      bpre[1] = a.best_f[s1];
#pragma unroll
      for (int u = 0; u < 8; ++u) {
        const int64_t k = min(u, m - 1);
        zpre[0][u] = a.Zt[k * S + s0];
        zpre[1][u] = a.Zt[k * S + s1];
      }
    }
    double tot[NQ];
    group_sum<NQ, WPR>(acc, red, tot, wv);
    if (tid < NQ) vv[tid] = tot[tid];
  }
  __syncthreads();
  if (tid < Q * Q) {
    const int i = tid / Q, j = tid % Q;
    const int ii = i > j ? i : j, jj = i > j ? j : i;
    sqq[i * Q + j] = ys2 * (sqq[i * Q + j] - vv[ii * (ii + 1) / 2 + jj]);
  }
  if (tid < Q) mu[tid] = a.y_mean + ys * (a.c + pv[tid * (n_b + 1)]);
  // ---- Sigma_qb into lnew[:, :n_b] (and a copy in dsqb for the joint mode)
  if (lb_lds) {
    if (tid < lay.lb_n) lbs[tid] = lbv;
    for (int e = tid + TPR; e < lay.lb_n; e += TPR) lbs[e] = a.Lb[e];
  }
  for (int e = tid; e < Q * n_b; e += TPR) {
    const int i = e / n_b, kb = e % n_b;
    const double sqb = ys2 * (lnew[i * m + kb] - pv[i * (n_b + 1) + 1 + kb]);
    lnew[i * m + kb] = sqb;
    if (joint) dsqb[e] = sqb;
  }
  __syncthreads();

  // Cached root (a.Lb): one substitution, then the q x q Schur block's
  // Cholesky with psd_safe_cholesky's jitter escalation.  Joint mode (the
  // reference's fallback to sampling from the joint posterior's Cholesky): the
  // jitter j_t of try t goes on the whole (n_b + q) x (n_b + q) diagonal, so try
  // t uses the baseline factor Lb_t = chol(Sigma_bb + j_t I) (a.Lb_levels, where
  // bit t of a.lb_levels_mask says it exists) and redoes the substitution.
  const double* Lb = a.Lb;
  int st_bits = 0;
  for (int t = 0; t <= (joint ? a.max_tries : 0); ++t) {
    if (joint) {
      if (!((a.lb_levels_mask >> t) & 1)) continue;  // the baseline block fails too
      Lb = a.Lb_levels + (int64_t)t * n_b * n_b;
      if (t > 0) {
        for (int e = tid; e < Q * n_b; e += TPR) lnew[(e / n_b) * m + e % n_b] = dsqb[e];
        __syncthreads();
      }
    }
    // ---- Lbl = Sigma_qb Lb^-T: forward substitution ---------------------
    if (lb_lds) solve16<Q, false, sizeof(TV) == 4>(lbs, n_b, lnew, m, lnew, m, wv, WPR);
    else solve_any<Q, false, sizeof(TV) == 4>(Lb, n_b, lnew, m, lnew, m, wv, WPR);
    __syncthreads();

    // ---- Schur complement and its Cholesky --------------------------------
    if (tid < Q * Q) {
      const int i = tid / Q, j = tid % Q;
      double s = 0.0;
#pragma unroll 4
      for (int kb = 0; kb < n_b; ++kb) s = fma(lnew[i * m + kb], lnew[j * m + kb], s);
      gA[i * Q + j] = sqq[i * Q + j] - s;  // gA used as scratch for the Schur block
    }
    __syncthreads();
    if (wv == 0) {
      int st = 0;
      bool ok = false;
      const int i = min(lane, Q - 1);
      double ar[Q], l[Q];
      bool mine = false;
#pragma unroll
      for (int j = 0; j < Q; ++j) {
        ar[j] = gA[i * Q + j];
        mine |= ar[j] != ar[j];
      }
      const bool has_nan = __ballot(mine) != 0;
      const int first = joint ? t : 0, last = joint ? t : a.max_tries;
      for (int attempt = first; attempt <= last && !has_nan; ++attempt) {
        const double jit = attempt == 0 ? 0.0 : a.jitter * pow(10.0, (double)(attempt - 1));
        ok = small_chol<Q>(ar, jit, i, l);
        if (ok) {
          if (attempt > 0) st |= BTA_STATUS_JITTER;
          break;
        }
      }
      if (has_nan) st |= BTA_STATUS_NAN;
      else if (!ok) st |= BTA_STATUS_NOT_PSD;
      if (lane < Q)
#pragma unroll
        for (int j = 0; j < Q; ++j) lbr[i * Q + j] = !ok ? NAN : j <= i ? l[j] : 0.0;
      if (lane == 0) scal[0] = (double)st;
    }
    __syncthreads();
    st_bits = (int)scal[0];
    if (!joint || !(st_bits & BTA_STATUS_NOT_PSD) || (st_bits & BTA_STATUS_NAN)) break;
    __syncthreads();  // every thread has read scal[0] before the next try rewrites it
  }
  if (joint && a.lb_levels_mask == 0 && tid == 0) {  // no baseline factor at any jitter
    scal[0] = (double)BTA_STATUS_NOT_PSD;
    for (int i = 0; i < Q * Q; ++i) lbr[i] = NAN;
  }
  __syncthreads();
  for (int e = tid; e < Q * Q; e += TPR) {
    const int i = e / Q, j = e % Q;
    lnew[i * m + n_b + j] = lbr[i * Q + j];
  }
  __syncthreads();

  // ---- samples, log improvement, fat-max over q ---------------------------
  // The per-sample transcendental arithmetic runs in TM: FP64 in the FP64
  // mode, FP32 in the mixed modes (samples and best_f stay FP64).
  typedef TV TM;
  const double tr = a.tau_relu, tm = a.tau_max, rtr = 1.0 / tr, rtm = 1.0 / tm;
  bool bad = false;
  double lmax = -INFINITY;  // this thread's max of u over its samples
  // y -> log improvement -> fat-max -> u[s], and the per-sample adjoint G[s]
  auto sample_tail = [&](const int s, const double bf, const double(&y)[Q]) {
    double v[Q], dv[Q];
    double M = -INFINITY;
#pragma unroll
    for (int i = 0; i < Q; ++i) {
      bad |= !isfinite(y[i]);
      log_fatplus_grad<TM>(y[i] - bf, tr, rtr, &v[i], &dv[i]);
      M = fmax(M, v[i]);
    }
    if constexpr (sizeof(TM) == 4) {
      TM P = 0, sdp = 0, dp[Q];
      int nties = 0;
#pragma unroll
      for (int i = 0; i < Q; ++i) {
        const TM z = (TM)((M - v[i]) * rtm);
        const TM den = (TM)2 + (TM)2 * z + z * z;
        P += div_tm((TM)2, den);
        dp[i] = div_tm((TM)-2 * ((TM)2 + (TM)2 * z), den * den);
        sdp += dp[i];
        nties += (v[i] == M);
      }
      const double u = M + tm * (double)log(P);
      uu[s] = u;
      lmax = fmax(lmax, u);
      const TM cm = div_tm((TM)1 + div_tm(sdp, P), (TM)nties);
#pragma unroll
      for (int i = 0; i < Q; ++i) {
        const TM du = (v[i] == M ? cm : (TM)0) - div_tm(dp[i], P);
        G[i * S + s] = (double)du * dv[i];
      }
    } else {
      double P = 0.0, sdp = 0.0, dp[Q], nties = 0.0;
#pragma unroll
      for (int i = 0; i < Q; ++i) {
        const double z = (M - v[i]) * rtm;
        const double rden = div_normal(1.0, fma(z, z, fma(2.0, z, 2.0)));
        P = fma(2.0, rden, P);
        dp[i] = -4.0 * (1.0 + z) * rden * rden;
        sdp += dp[i];
        nties += v[i] == M ? 1.0 : 0.0;
      }
      const double u = M + tm * log_pos(P);
      uu[s] = u;
      lmax = fmax(lmax, u);
      const double rP = div_normal(1.0, P);
      const double cm = div_normal(fma(sdp, rP, 1.0), nties);
#pragma unroll
      for (int i = 0; i < Q; ++i)
        G[i * S + s] = ((v[i] == M ? cm : 0.0) - dp[i] * rP) * dv[i];
    }
  };
  // Each thread carries the samples s0 and s0 + TPR through the products: the
  // rows of [Lbl | Lbr] (LDS) and the base samples are read eight columns at a
  // time at clamped indices, so that every read issues before the products;
  // the products skip the columns past m.
  for (int s0 = tid; s0 < S; s0 += 2 * TPR) {
    const bool two = s0 + TPR < S;
    const int s1 = two ? s0 + TPR : s0;
    const bool pre = ZPRE && s0 == tid;
    double bf0, bf1;
    if (pre) {
      bf0 = bpre[0];
      bf1 = bpre[1];
    } else {
      bf0 = a.best_f[s0];
      bf1 = a.best_f[s1];
    }
    double y0[Q], y1[Q];
#pragma unroll
    for (int i = 0; i < Q; ++i) y0[i] = y1[i] = mu[i];
    for (int k0 = 0; k0 < m; k0 += 8) {
      double lc[Q][8], z0[8], z1[8];
      if (pre && k0 == 0) {
#pragma unroll
        for (int u = 0; u < 8; ++u) {
          z0[u] = zpre[0][u];
          z1[u] = zpre[1][u];
        }
      } else {
#pragma unroll
        for (int u = 0; u < 8; ++u) {
          const int64_t k = k0 + u < m ? k0 + u : m - 1;
          z0[u] = a.Zt[k * S + s0];
          z1[u] = a.Zt[k * S + s1];
        }
      }
#pragma unroll
      for (int u = 0; u < 8; ++u) {
        const int k = k0 + u < m ? k0 + u : m - 1;
#pragma unroll
        for (int i = 0; i < Q; ++i) lc[i][u] = lnew[i * m + k];
      }
#pragma unroll
      for (int u = 0; u < 8; ++u)
        if (k0 + u < m)
#pragma unroll
          for (int i = 0; i < Q; ++i) {
            y0[i] = fma(lc[i][u], z0[u], y0[i]);
            y1[i] = fma(lc[i][u], z1[u], y1[i]);
          }
    }
    // one or two candidates leave room between the dependent operations of a sample:
    // its partner's go there (a thread without one repeats its own)
    if (sizeof(TM) == 8 && Q <= 2 && __any(two)) {
      sample_tail(s0, bf0, y0);
      sample_tail(s1, bf1, y1);
    } else {
      sample_tail(s0, bf0, y0);
      if (two) sample_tail(s1, bf1, y1);
    }
  }
  if (bad) scal[1] = 1.0;  // every writer stores the same value

  // ---- logmeanexp over samples (each thread reads back only its own u[s]
  // and G[s] until the next barrier) ----------------------------------------
  const double Mu = group_max1<WPR>(lmax, red, wv);
  double lsum[1] = {0.0};
  for (int s = tid; s < S; s += TPR) {  // uu keeps exp(u - max) for the adjoint
    const double e = sizeof(TM) == 4 ? exp(uu[s] - Mu) : exp_nonpos(uu[s] - Mu);
    uu[s] = e;
    lsum[0] += e;
  }
  double tsum[1];
  group_sum<1, WPR>(lsum, red, tsum, wv);
  auto write_value = [&]() {
    if (tid == TPR - 1 && live) {
      a.value[b] = Mu + log(tsum[0]) - log((double)S);
      int st = (int)scal[0];
      if (scal[1] != 0.0) st |= BTA_STATUS_NAN;
      a.status[b] = st;
    }
  };
  if (!a.grad) {
    write_value();
    return;
  }

  // ---- dmu, d[Lbl | Lbr] = (w G)^T Z with the logmeanexp weights w --------
  // per-thread accumulators while m <= MREG (FP32 samples; in FP64 the registers they
  // take cost more than the second pass over G)
  constexpr bool f32 = sizeof(TM) == 4;
  constexpr int MREG = 32 / Q - 1;
  if (f32 && m <= MREG) {
    if constexpr (f32) {
    constexpr int NV = Q * (MREG + 1);
    double acc[NV];
#pragma unroll
    for (int e = 0; e < NV; ++e) acc[e] = 0.0;
    auto accum = [&](const int s, const double(&z)[MREG]) {
      const double w = uu[s] / tsum[0];
      double gw[Q];
#pragma unroll
      for (int i = 0; i < Q; ++i) {
        gw[i] = G[i * S + s] * w;
        acc[i * (MREG + 1) + MREG] += gw[i];
      }
#pragma unroll
      for (int k = 0; k < MREG; ++k) {
        if (k < m) {
#pragma unroll
          for (int i = 0; i < Q; ++i)
            acc[i * (MREG + 1) + k] = fma(gw[i], z[k], acc[i * (MREG + 1) + k]);
        }
      }
    };
    // samples s and s + TPR per pass, the base samples of both loaded ahead of
    // the products (uniform branches); the sums run in sample order as before
    for (int s = tid; s < S; s += 2 * TPR) {
      const bool two = s + TPR < S;
      const int s2 = two ? s + TPR : s;
      double z[MREG], z2[MREG];
#pragma unroll
      for (int k = 0; k < MREG; ++k)
        if (k < m) {
          z[k] = a.Zt[(int64_t)k * S + s];
          z2[k] = a.Zt[(int64_t)k * S + s2];
        }
      accum(s, z);
      if (two) accum(s2, z2);
    }
    {
      int e;
      const double sw = wave_sum_spread<NV>(acc, &e);
      if (e >= 0) red[wv * 64 + e] = sw;
    }
    __syncthreads();
    for (int e = tid; e < Q * (m + 1); e += TPR) {
      const int i = e / (m + 1), k = e % (m + 1);
      const int idx = i * (MREG + 1) + (k == m ? MREG : k);
      double tot = red[idx];
#pragma unroll
      for (int w = 1; w < WPR; ++w) tot += red[w * 64 + idx];
      if (k == m) dmu[i] = tot;
      else dlnew[i * m + k] = k < n_b + i + 1 ? tot : 0.0;
    }
    __syncthreads();
    }
  } else {
  for (int s = tid; s < S; s += TPR) {
    const double w = uu[s] / tsum[0];
#pragma unroll
    for (int i = 0; i < Q; ++i) G[i * S + s] *= w;
  }
  __syncthreads();

  // wide baselines: wave w sums the columns w, w + WPR, .. (four at a time, with all
  // rows i: the base samples are read once and the wave sums share their exchanges);
  // column m, the means, takes base samples of 1
  for (int k0 = wv; k0 <= m; k0 += 4 * WPR) {
    double acc[4 * Q];
#pragma unroll
    for (int e = 0; e < 4 * Q; ++e) acc[e] = 0.0;
#pragma unroll 4
    for (int s = lane; s < S; s += 64) {
      double z[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const int k = k0 + u * WPR;
        z[u] = a.Zt[(int64_t)min(k, m - 1) * S + s];
        z[u] = k < m ? z[u] : 1.0;
      }
#pragma unroll
      for (int i = 0; i < Q; ++i) {
        const double gi = G[i * S + s];
#pragma unroll
        for (int u = 0; u < 4; ++u) acc[u * Q + i] = fma(gi, z[u], acc[u * Q + i]);
      }
    }
    int e;
    const double tot = wave_sum_spread<4 * Q>(acc, &e);
    const int i = e % Q, k = k0 + e / Q * WPR;
    if (e >= 0 && k <= m) {
      if (k == m) dmu[i] = tot;
      else dlnew[i * m + k] = k < n_b + i + 1 ? tot : 0.0;  // (upper part of Lbr: none)
    }
  }
  __syncthreads();
  }

  // ---- Cholesky backward of Lbr (torch's formula), gA symmetric ----------
  // by the restart's first wave: lane (i, j) forms an entry of tril(L^T dL), lane j a
  // column of Y, lane r a row of gA; T and Y pass through red.  (Where a rounded
  // product is added rather than fused, it is the rounding the one-lane form had.)
  if (wv == 0) {
    double* Ts = red;
    double* Ys = red + 64;
    const int e = min(lane, Q * Q - 1), ti = e / Q, tj = e % Q, c = min(lane, Q - 1);
    double t = 0.0;
#pragma unroll
    for (int k = 0; k < Q; ++k) t = fma(lbr[k * Q + ti], dlnew[k * m + n_b + tj], t);
    Ts[e] = tj <= ti ? t : 0.0;
    const double rc = 1.0 / lbr[c * Q + c];
    double rd[Q], y[Q];
#pragma unroll
    for (int i = 0; i < Q; ++i) rd[i] = lane_bcast(rc, i);
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    // Y = L^-T Mm, Mm = the symmetric half of T: back substitution per column
#pragma unroll
    for (int i = Q - 1; i >= 0; --i) {
      double s = 0.5 * (i >= c ? Ts[i * Q + c] : Ts[c * Q + i]);
#pragma unroll
      for (int k = i + 1; k < Q; ++k) {
        const double p = -lbr[k * Q + i];
        s = k == i + 1 && i == c ? s + fma(p, y[k], 0.0) : fma(p, y[k], s);
      }
      y[i] = i ? s * rd[i] : s;  // row 0 is scaled where it is used
    }
#pragma unroll
    for (int i = 0; i < Q; ++i) Ys[i * Q + c] = y[i];
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    // gA = Y L^-1: x L = y for each row
#pragma unroll
    for (int j = Q - 1; j >= 0; --j) {
      double s = Ys[c * Q + j];
      if (j + 1 < Q) {
        const double l = lbr[(j + 1) * Q + j];
        s = c == 0 ? fma(s, rd[0], fma(-y[j + 1], l, 0.0)) : fma(-y[j + 1], l, s);
      } else {
        s = c == 0 ? s * rd[0] : s;
      }
#pragma unroll
      for (int k = j + 2; k < Q; ++k) s = fma(-y[k], lbr[k * Q + j], s);
      y[j] = s * rd[j];
    }
    if (lane < Q)
#pragma unroll
      for (int j = 0; j < Q; ++j) gA[c * Q + j] = y[j];
  }
  __syncthreads();
  // dLbl -= 2 gA Lbl  (Schur = Sigma_qq - Lbl Lbl^T)
  for (int e = tid; e < Q * n_b; e += TPR) {
    const int i = e / n_b, kb = e % n_b;
    double s = 0.0;
#pragma unroll
    for (int j = 0; j < Q; ++j) s += gA[i * Q + j] * lnew[j * m + kb];
    dlnew[i * m + kb] -= 2.0 * s;
  }
  __syncthreads();
  // ---- dSigma_qb = dLbl Lb^-1: back substitution ---------------------------
  if (lb_lds) solve16<Q, true, sizeof(TV) == 4>(lbs, n_b, dlnew, m, dsqb, n_b, wv, WPR);
  else solve_any<Q, true, sizeof(TV) == 4>(Lb, n_b, dlnew, m, dsqb, n_b, wv, WPR);
  __syncthreads();

  // ---- dV = gq V with gq = -2 s^2 gA: the q x q block for the gradient stage
  write_value();  // (here, where no barrier waits for its logarithms)
  if (!live) return;
  for (int e = tid; e < Q * Q; e += TPR) a.gq[r0 * Q + e] = -2.0 * ys2 * gA[e];
  for (int e = tid; e < Q * (n_b + 1); e += TPR) {
    const int i = e / (n_b + 1), k = e % (n_b + 1);
    a.dext[(r0 + i) * (n_b + 1) + k] = k == 0 ? ys * dmu[i] : -ys2 * dsqb[i * n_b + k - 1];
  }
  // ---- direct input gradient through K(X, X) and K(X, X_b) (scaled), from
  // the radial factors hh computed with the kernel values ------------------
  for (int e = tid; e < Q * d; e += TPR) {
    const int i = e / d, j = e % d;
    const double xij = xq[i * MC_MAXD + j];
    double acc = 0.0;
    for (int i2 = 0; i2 < Q; ++i2)
      acc -= 2.0 * ys2 * gA[i * Q + i2] * hh[i * m + i2] * (xij - xq[i2 * MC_MAXD + j]);
#pragma unroll 4
    for (int kb = 0; kb < n_b; ++kb)
      acc -= ys2 * dsqb[i * n_b + kb] * hh[i * m + Q + kb] * (xij - a.bs[kb * d + j]);
    a.dxs_extra[(r0 + i) * d + j] = acc;
  }
}

// One launch for the adjoint GEMM U = V L^-1 and the MC stage uses the first
// NR McLayout areas of the GEMM's LDS ring (64-column tiles; NR areas stay
// within MC_LDS_MAX).
constexpr int FUSED_LDS = H2Mid::STAGES * H2Mid::STAGE;
static_assert(MC_LDS_MAX <= (size_t)FUSED_LDS, "MC layout must fit the fused ring");

// dX = (sum of the column-tile partials + direct term) / lengthscale.
struct FinishArgs {
  const double* Dpart;
  int nct;
  int64_t R;
  int d;
  const double* extra;
  const double* ls;
  double* dX;
};

// Every launch argument of one model's value(+grad) step, and its workspace
// plan.  Built by qlognei_step_args from the caller's buffers.
struct StepArgs {
  int64_t b, R, R_pad, np;
  int q, covar_mode;            // covar_mode: 0 FP64, 1 FP32, 2 FP16 planes
  bool f32, split, grad;
  QsCovarArgs c;
  H2Args fwd, adj;              // split mode: V = K_x L^-T, U = V L^-1
  int gemm_flags;               // FP64 / mixed_f32 products through gemm()
  void* kx;
  void* vt;
  const void* linv;
  McArgs mc;
  QsGradArgs g;
  FinishArgs fin;
};

size_t qlognei_ws_bytes(const bta_gp_model* m, const bta_qlognei_state* st, int64_t b);
// Checks the arguments of one step and fills A (nothing is launched).
int qlognei_step_args(const bta_gp_model* m, const bta_qlognei_state* st, const double* X,
                      int64_t b, double* value, double* grad, int* status, void* ws,
                      size_t ws_bytes, StepArgs& A);

}  // namespace bta
