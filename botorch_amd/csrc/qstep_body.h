// Device bodies of the qLogNEI step's elementwise stages (the algorithm is
// described at the top of qstep.hip).  Each body works on the tile or lanes it
// is given, so the same code runs as one model's kernel (qstep.hip) and as the
// per-model share of a launch over many models (the batched step in
// qlognei.hip).
#pragma once
#include "bta_common.h"
#include "kernels.h"

#include <type_traits>

namespace bta {

constexpr int QS_RT = 64;           // rows per block (16 per wave)
constexpr int QS_CT = QS_COL_TILE;  // columns (training points) per block
constexpr int QS_MAXQ = 8;

__device__ __forceinline__ v4d mfma64(double a, double b, v4d c) {
  return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
}

// The 64 training points of a column tile, their coordinates from registers
// (qs_load_t) and their squared norms, one copy of these per wave: no barrier between
// writing and reading them.
template <int KD>
struct QsT {
  double tc[QS_CT][4 * KD + 1];
  double tn2[4][QS_CT];
};

template <int KD>
__device__ __forceinline__ void qs_load_t(double (&tv)[KD], const double* T, int n, int d,
                                          int c0) {
  constexpr int MD = 4 * KD;
#pragma unroll
  for (int t = 0; t < KD; ++t) {
    const int e = threadIdx.x + 256 * t, c = e / MD, j = e % MD;
    tv[t] = (j < d && c0 + c < n) ? T[(int64_t)(c0 + c) * d + j] : 0.0;
  }
}
template <int KD>
__device__ __forceinline__ void qs_store_t(QsT<KD>& sm, const double (&tv)[KD]) {
#pragma unroll
  for (int t = 0; t < KD; ++t) {
    const int e = threadIdx.x + 256 * t;
    sm.tc[e / (4 * KD)][e % (4 * KD)] = tv[t];
  }
}
// after the barrier that follows qs_store_t
template <int KD>
__device__ __forceinline__ void qs_norms(QsT<KD>& sm) {
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  double s = 0.0;
#pragma unroll
  for (int j = 0; j < 4 * KD; ++j) s = fma(sm.tc[lane][j], sm.tc[lane][j], s);
  sm.tn2[wv][lane] = s;
}

// sum over the four 16-lane groups (same lane % 16)
__device__ __forceinline__ double sum_groups(double v) {
  v += __shfl_xor(v, 16, 64);
  v += __shfl_xor(v, 32, 64);
  return v;
}

template <typename TO>
struct alignas(16) QsKStage {
  TO k[QS_RT][QS_CT + 16 / (int)sizeof(TO)];
};

// mode: 0 = FP64 K, 1 = FP32 K, 2 = FP16 hi/lo planes of K * kscale
// One 64-row x 64-column tile (column tile ct, row tile rt) of the covariance
// stage; 256 threads.
template <int KD, int MODE, int KIND>
__device__ __forceinline__ void qstep_covar_body(const QsCovarArgs& a, const int ct,
                                                 const int rt) {
  typedef typename std::conditional<MODE == 0, double,
                                    typename std::conditional<MODE == 1, float,
                                                              _Float16>::type>::type TO;
  __shared__ QsT<KD> sm;
  __shared__ QsKStage<TO> ks[MODE == 2 ? 2 : 1];
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
  const int l16 = lane & 15, g = lane >> 4;
  const int d = a.d, ne = a.ne, n = (int)a.n, R = (int)a.R;  // (grid extents are 64 x smaller)
  const int c0 = ct * QS_CT, r0 = rt * QS_RT;
  const int r0w = r0 + wv * 16;
  const int rl = r0w + l16;  // this lane's row as B operand / D column
  // Every global load of the block is issued before the staging barrier: T, the
  // raw row coordinates and the first 16 columns of E (all of them for ne <= 16).
  double tv[KD], xr[KD], xc[KD], xl[KD];
  qs_load_t<KD>(tv, a.T, n, d, c0);
  const double* xrow = a.X + (int64_t)min(rl, R - 1) * d;
  const double* E = a.E + (int64_t)c0 * ne + l16;
#pragma unroll
  for (int s = 0; s < KD; ++s) {
    const int j = 4 * s + g;
    const bool ok = j < d && rl < R;
    xr[s] = ok ? xrow[j] : 0.0;
    xc[s] = ok ? a.center[j] : 0.0;
    xl[s] = ok ? a.ls[j] : 1.0;
  }
  double ev[4][4];
#pragma unroll
  for (int cb = 0; cb < 4; ++cb)
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int c = cb * 16 + g + 4 * q;
      ev[cb][q] = (l16 < ne && c0 + c < n) ? E[c * ne] : 0.0;
    }
  qs_store_t<KD>(sm, tv);
  __syncthreads();
  qs_norms<KD>(sm);

  // scaled row coordinates: lane (g, l16) holds x[rl][4s + g]
  double xb[KD];
  double xn2 = 0.0;
#pragma unroll
  for (int s = 0; s < KD; ++s) {
    const int j = 4 * s + g;
    const double v = (xr[s] - xc[s]) / xl[s];
    xb[s] = v;
    xn2 = fma(v, v, xn2);
    if (ct == 0 && j < d) a.xs_out[(int64_t)rl * d + j] = v;
  }
  xn2 = sum_groups(xn2);

  // K^T blocks: kv[cb][q] = K[rl][c0 + cb*16 + g + 4q]
  double kv[4][4];
#pragma unroll
  for (int cb = 0; cb < 4; ++cb) {
    v4d cr = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
    for (int s = 0; s < KD; ++s) cr = mfma64(sm.tc[cb * 16 + l16][4 * s + g], xb[s], cr);
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int cl = cb * 16 + g + 4 * q;
      const double r2 = fmax(sm.tn2[wv][cl] + xn2 - 2.0 * cr[q], 0.0);
      double k = kern_value_k<KIND>(r2, a.s);
      k = (c0 + cl < n && rl < R) ? k : 0.0;
      kv[cb][q] = k;
      if (MODE == 2) {
        // kscale is a power of two: scaling after the FP32 rounding is exact
        const float x = (float)k * a.kscale;
        const _Float16 h = (_Float16)x;
        ks[0].k[wv * 16 + l16][cl] = h;
        ks[MODE == 2 ? 1 : 0].k[wv * 16 + l16][cl] = (_Float16)((x - (float)h) * 2048.0f);
      } else {
        ks[0].k[wv * 16 + l16][cl] = (TO)k;
      }
    }
  }
  __syncthreads();
  // coalesced 16-byte row stores of the K tile (planes)
  {
    constexpr int V = 16 / (int)sizeof(TO);  // elements per 16-byte chunk
    constexpr int CPR = QS_CT / V;           // chunks per row
    const int64_t o0 = (int64_t)(r0 + tid / CPR) * a.ldk + c0 + tid % CPR * V;
#pragma unroll
    for (int e0 = 0; e0 < QS_RT * CPR; e0 += 256) {
      const int r = (tid + e0) / CPR, cc = tid % CPR * V;
      const int64_t o = o0 + e0 / CPR * a.ldk;
      *(int4*)((TO*)a.K + o) = *(const int4*)&ks[0].k[r][cc];
      if (MODE == 2) *(int4*)(a.Klo + o) = *(const int4*)&ks[MODE == 2 ? 1 : 0].k[r][cc];
    }
  }
  // Ppart[r][j][ct] = sum_c K[r][c] E[c][j] in chunks of 16 columns j
  const int64_t nct = a.n_pad / QS_CT;
  for (int j0 = 0; j0 < ne; j0 += 16) {
    const int jj = j0 + l16;
    v4d p = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
    for (int cb = 0; cb < 4; ++cb)
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int c = cb * 16 + g + 4 * q;
        const double e =
            j0 == 0 ? ev[cb][q] : ((jj < ne && c0 + c < n) ? E[c * ne + j0] : 0.0);
        p = mfma64(kv[cb][q], e, p);
      }
    // D layout: lane (g, l16) reg q = P[r0w + g + 4q][jj]
    double* pp = a.Ppart + ((int64_t)(r0w + g) * ne + jj) * nct + ct;
    const int64_t step = 4 * (int64_t)ne * nct;
#pragma unroll
    for (int q = 0; q < 4; ++q)
      if (jj < ne && r0w + g + 4 * q < R) pp[q * step] = p[q];
  }
}

// U rows that 16 rows of a wave can mix, in steps of 4: 28 rows at q = 7.
constexpr int QS_KU = 7;
constexpr int QS_E_LDS = 16;  // columns of E staged in LDS (the rest is read per block)

// One tile of the gradient stage (column tile ct, row tile rt); 256 threads.
// A tile is ~80 matrix products a wave, so what it waits for shows: every load of the
// tile (T and E through LDS, the U rows, the restart blocks and dext in the lanes of
// their matrix operands) is issued before the one barrier.  With the loads beside each
// product a 64-point model's launch took 14.1 us, now 8.7 us; 2048 points, 2048 rows:
// 28.4 -> 23.7 us; 16384 points, 8192 rows: 1053 -> 821 us.
template <int KD, typename TU, int KIND>
__device__ __forceinline__ void qstep_grad_body(const QsGradArgs& a, const int ct,
                                                const int rt) {
  constexpr int NB = (4 * KD + 1 + 15) / 16;  // 16-column blocks of [T | 1]
  __shared__ QsT<KD> sm;
  __shared__ double es[QS_CT][QS_E_LDS + 1];
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
  const int l16 = lane & 15, g = lane >> 4;
  const int d = a.d, q = a.q, ne = a.ne;
  const int R = (int)a.R, n = (int)a.n;  // (both grid extents are 64 times smaller)
  const int c0 = ct * QS_CT, r0w = rt * QS_RT + wv * 16;
  const int rl = r0w + l16;
  const bool rvalid = rl < R;
  const int64_t rc = rvalid ? rl : R - 1;  // in-bounds row of this lane
  // U rows feeding this wave's rows: whole restarts [kr0, kr1)
  const int kr0 = r0w - r0w % q;
  const int kr1 = min(((r0w + 15) / q + 1) * q, R);
  const int ku = kr1 > kr0 ? (kr1 - kr0 + 3) / 4 : 0;
  const int rblk = rl - rl % q;  // first row of this lane's restart

  // ---- loads ----------------------------------------------------------------
  double tv[KD], ev[4];
  qs_load_t<KD>(tv, a.T, n, d, c0);
  const int ec = tid >> 2;
#pragma unroll
  for (int t = 0; t < 4; ++t) {
    const int j = 4 * t + (tid & 3);
    ev[t] = (j < ne && c0 + ec < n) ? a.E[(int64_t)(c0 + ec) * ne + j] : 0.0;
  }
  double xb[KD], db[4], mb[QS_KU];
#pragma unroll
  for (int s = 0; s < KD; ++s) {
    const int j = 4 * s + g;
    xb[s] = (j < d && rvalid) ? a.xs[rc * d + j] : 0.0;
  }
#pragma unroll
  for (int s = 0; s < 4; ++s) {
    const int j = 4 * s + g;
    db[s] = (j < ne && rvalid) ? a.dext[rc * ne + j] : 0.0;
  }
  TU uv[QS_KU][4];
  const TU* U = (const TU*)a.U + c0 + l16;
#pragma unroll
  for (int s = 0; s < QS_KU; ++s) {
    const int u = kr0 + 4 * s + g;
    mb[s] = 0.0;
    if (s < ku) {
#pragma unroll
      for (int cb = 0; cb < 4; ++cb) uv[s][cb] = U[(int64_t)min(u, R - 1) * a.ldu + cb * 16];
      // u in this lane's restart [rblk, rblk + q) (rows beyond R never are)
      if (rvalid && u >= rblk && u < rblk + q) mb[s] = a.gq[rc * q + (u - rblk)];
    }
  }
  qs_store_t<KD>(sm, tv);
#pragma unroll
  for (int t = 0; t < 4; ++t) es[ec][4 * t + (tid & 3)] = ev[t];
  __syncthreads();
  qs_norms<KD>(sm);
  double xn2 = 0.0;
#pragma unroll
  for (int s = 0; s < KD; ++s) xn2 = fma(xb[s], xb[s], xn2);
  xn2 = sum_groups(xn2);

  v4d dacc[NB];
#pragma unroll
  for (int nb = 0; nb < NB; ++nb) dacc[nb] = (v4d){0.0, 0.0, 0.0, 0.0};
#pragma unroll
  for (int cb = 0; cb < 4; ++cb) {
    const int ca = c0 + cb * 16 + l16;  // A-operand column
    v4d cr = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
    for (int s = 0; s < KD; ++s) cr = mfma64(sm.tc[cb * 16 + l16][4 * s + g], xb[s], cr);
    // G^T[c][r] = sum_j E[c][j] dext[r][j] + sum_u U[u][c] M[u][r]
    v4d ga = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
    for (int s = 0; s < 4; ++s)
      if (4 * s < ne) ga = mfma64(es[cb * 16 + l16][4 * s + g], db[s], ga);
    for (int j0 = QS_E_LDS; j0 < ne; j0 += 4) {
      const int j = j0 + g;
      const double ea = (j < ne && ca < n) ? a.E[(int64_t)ca * ne + j] : 0.0;
      const double de = (j < ne && rvalid) ? a.dext[rc * ne + j] : 0.0;
      ga = mfma64(ea, de, ga);
    }
#pragma unroll
    for (int s = 0; s < QS_KU; ++s)
      if (s < ku) {
        const bool ok = kr0 + 4 * s + g < kr1 && ca < n;
        ga = mfma64(ok ? (double)uv[s][cb] : 0.0, mb[s], ga);
      }
    // w^T[c][r] = -G h(r^2); then [T | 1]-contraction over c
#pragma unroll
    for (int qq = 0; qq < 4; ++qq) {
      const int cl = cb * 16 + g + 4 * qq;
      const double r2 = fmax(sm.tn2[wv][cl] + xn2 - 2.0 * cr[qq], 0.0);
      double w = -ga[qq] * kern_grad_factor_k<KIND>(r2, a.s);
      w = (c0 + cl < n && rvalid) ? w : 0.0;
#pragma unroll
      for (int nb = 0; nb < NB; ++nb) {
        const int j = nb * 16 + l16;
        const double tb = j < d ? sm.tc[cl][j] : (j == d ? 1.0 : 0.0);
        dacc[nb] = mfma64(w, tb, dacc[nb]);
      }
    }
  }
  // D layout: lane (g, l16) reg qq = S[r0w + g + 4qq][nb*16 + l16], S = w [T | 1]
  const int src = g * 16 + (d & 15);
#pragma unroll
  for (int qq = 0; qq < 4; ++qq) {
    double sw = 0.0;  // sum_c w[r][c], held in column d
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) {
      const double v = __shfl(dacc[nb][qq], src, 64);
      if (nb == d / 16) sw = v;
    }
    const int64_t r = r0w + g + 4 * qq;
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) {
      const int j = nb * 16 + l16;
      if (j < d && r < R)
        a.Dpart[((int64_t)ct * a.R + r) * d + j] = a.xs[r * d + j] * sw - dacc[nb][qq];
    }
  }
}

// Four lanes per element, each summing every fourth partial (8 loads in
// flight), then combined in a fixed order: deterministic.  gid: the thread's
// index over the 4 R d lanes of the stage.
__device__ __forceinline__ void qstep_finish_body(const double* __restrict__ Dpart, int nct,
                                                  int64_t R, int d,
                                                  const double* __restrict__ extra,
                                                  const double* __restrict__ ls,
                                                  double* __restrict__ dX, const int64_t gid) {
  const int64_t e = gid >> 2;
  const int part = (int)(gid & 3);
  const int64_t tot = R * d;
  double acc = 0.0;
  if (e < tot) {
#pragma unroll 8
    for (int t = part; t < nct; t += 4) acc += Dpart[(int64_t)t * tot + e];
  }
  acc += __shfl_xor(acc, 1, 64);
  acc += __shfl_xor(acc, 2, 64);
  if (part == 0 && e < tot) dX[e] = (acc + (extra ? extra[e] : 0.0)) / ls[(int)(e % d)];
}

}  // namespace bta
