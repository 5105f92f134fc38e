// GP posterior moments over batch x mq points and their adjoint.
//
//   K_x = s k(xs, X_train);  V = K_x L^-T;  mean = y_mean + y_std (c + K_x alpha)
//   covar = y_std^2 (k(xs, xs) - V V^T)  per batch element
//
// Rows: up to POST_SMALL_MQ points per batch element the rows of all elements
// lie one after another (row b mq + i) and only their total is padded, to the
// GEMM's 128-row tile; above it every element's rows are padded to a multiple of
// 64, the tile edge of the mq x mq products.  Padding each element to 64 rows
// at every mq cost 64 / mq of all the work: 256 x 4 points against n = 2048 took
// 5.5 ms for moments, samples and gradient on 16384 rows instead of 1024.
//
// Moments, three launches (the GEMM aside):
//   post_covar_kernel      xs, K_x and the 64-column partials of K_x alpha
//   post_cov_small_kernel  mq <= POST_SMALL_MQ: V V^T on MFMA for 16 consecutive
//                          rows, k(xs, xs), and all the outputs
//   post_cov_tiles_kernel, post_cov_joint_kernel  above: lower 32 x 32 or 128 x 64
//                          tiles of V V^T, the same epilogue, the upper triangle
//                          mirrored
// Adjoint: U = V L^-1 = K_x K^-1 (with xs and V kept from the moments' call, or K_x
// and V formed again: 120 of 520 us at 256 x 4 points and n = 2048), then
//   post_grad_kernel       g_rc = y_std dmean_r alpha_c - sum_j S_rj U_jc with
//                          S = y_std^2 (dC + dC^T), times dk/dxs, over a share
//                          of the columns
//   post_grad_finish_kernel sums the shares, adds the term through k(xs, xs)
// Distances are direct coordinate differences (no cancellation near training
// points).  All sums have a fixed order.
#include "bta_common.h"
#include "gemm.h"
#include "gemm_d.h"
#include "gemm_tile.h"
#include "gemm_w_body.h"
#include "kernels.h"

#include <algorithm>

namespace bta {

constexpr int POST_SMALL_MQ = 16;  // one MFMA block holds whole batch elements
constexpr int PC_ROWS = 16;        // rows per block of post_covar_kernel
constexpr int PC_MAXD = 32;
constexpr int PG_COLS = 256;       // columns per pass of post_grad_kernel

// Row p of the padded row layout -> its batch element and point; false in the
// padding.
struct PostRows {
  int64_t batch;
  int mq, mq_pad;
  __device__ __forceinline__ bool at(int64_t p, int64_t& bi, int& r) const {
    const uint32_t b = (uint32_t)p / (uint32_t)mq_pad;  // p < 2^31 (post_check)
    bi = b;
    r = (int)((uint32_t)p - b * (uint32_t)mq_pad);
    return bi < batch && r < mq;
  }
};

__device__ __forceinline__ double kern_any(int kind, double r2, double s) {
  return kind == BTA_KERNEL_MATERN52 ? kern_value_k<BTA_KERNEL_MATERN52>(r2, s)
                                     : kern_value_k<BTA_KERNEL_RBF>(r2, s);
}

struct PostCovarArgs {
  const double* X;  // batch x mq x d query points
  PostRows rows;
  const double *center, *ls, *T, *alpha;  // T: n x d scaled training inputs
  double* xs;    // R_pad x d scaled rows (zero in the padding)
  double* K;     // R_pad x n_pad
  double* part;  // R_pad x (n_pad / 64) partials of K alpha, or null
  int64_t n, n_pad;
  int d;
  double s;
};

// 16 rows x 256 columns per block: a thread keeps its training point in
// registers, the rows sit in LDS (broadcast reads), every store is a coalesced
// row segment.  The product with alpha, which a GEMM with a 64-row padded alpha
// took 100 us for at 1500 x 1000, rides on the kernel values.
template <int MD, int KIND>
__global__ __launch_bounds__(256) void post_covar_kernel(PostCovarArgs a) {
  __shared__ double xr[PC_ROWS * MD];
  const int d = a.d;
  const int64_t r0 = (int64_t)blockIdx.y * PC_ROWS;
  const int64_t c = (int64_t)blockIdx.x * 256 + threadIdx.x;
  for (int i = threadIdx.x; i < PC_ROWS * MD; i += 256) {
    const int64_t p = r0 + i / MD;
    const int j = i % MD;
    int64_t bi;
    int r;
    const bool ok = a.rows.at(p, bi, r) && j < d;
    const double v =
        ok ? (a.X[(bi * a.rows.mq + r) * d + j] - a.center[j]) / a.ls[j] : 0.0;
    xr[i] = v;
    if (blockIdx.x == 0 && j < d) a.xs[p * d + j] = v;
  }
  const bool cvalid = c < a.n;
  double t[MD];
#pragma unroll
  for (int j = 0; j < MD; ++j) t[j] = (cvalid && j < d) ? a.T[c * d + j] : 0.0;
  const double al = (a.part && cvalid) ? a.alpha[c] : 0.0;
  __syncthreads();
  double pr[PC_ROWS];
#pragma unroll
  for (int rr = 0; rr < PC_ROWS; ++rr) {
    const int64_t p = r0 + rr;
    int64_t bi;
    int r;
    double v = 0.0;
    if (cvalid && a.rows.at(p, bi, r)) {
      double r2 = 0.0;
#pragma unroll
      for (int j = 0; j < MD; ++j) {
        const double df = xr[rr * MD + j] - t[j];
        r2 = fma(df, df, r2);
      }
      v = kern_value_k<KIND>(r2, a.s);
    }
    if (c < a.n_pad) a.K[p * a.n_pad + c] = v;
    pr[rr] = v * al;
  }
  if (!a.part) return;
  int e;
  const double sum = wave_sum_spread<PC_ROWS>(pr, &e);
  const int64_t tile = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (e >= 0 && tile < a.n_pad / 64) a.part[(r0 + e) * (a.n_pad / 64) + tile] = sum;
}

template <int MD>
static void post_covar_k(const PostCovarArgs& a, int kind, dim3 g, hipStream_t s) {
  if (kind == BTA_KERNEL_MATERN52)
    hipLaunchKernelGGL((post_covar_kernel<MD, BTA_KERNEL_MATERN52>), g, dim3(256), 0, s, a);
  else
    hipLaunchKernelGGL((post_covar_kernel<MD, BTA_KERNEL_RBF>), g, dim3(256), 0, s, a);
}

static int post_covar(const PostCovarArgs& a, int kind, int64_t R_pad, hipStream_t s) {
  const dim3 g((unsigned)((a.n_pad + 255) / 256), (unsigned)(R_pad / PC_ROWS));
  switch ((a.d + 3) / 4) {
    case 1: post_covar_k<4>(a, kind, g, s); break;
    case 2: post_covar_k<8>(a, kind, g, s); break;
    case 3: post_covar_k<12>(a, kind, g, s); break;
    case 4: post_covar_k<16>(a, kind, g, s); break;
    case 5: post_covar_k<20>(a, kind, g, s); break;
    case 6: post_covar_k<24>(a, kind, g, s); break;
    case 7: post_covar_k<28>(a, kind, g, s); break;
    default: post_covar_k<32>(a, kind, g, s); break;
  }
  BTA_LAUNCH_CHECK("post_covar_kernel");
  return BTA_OK;
}

struct PostOutArgs {
  const double *V, *xs, *part;
  PostRows rows;
  int64_t n_pad;
  int d, kind;
  double s, y_mean, y_std, c;
  double *mean, *covar, *var;  // each may be null
};

// mean of padded row p from its partials, summed by the 16 lanes of a 16-lane
// group (every lane gets the total)
__device__ __forceinline__ double post_mean16(const PostOutArgs& a, int64_t p) {
  const int nt = (int)(a.n_pad / 64);
  const double* q = a.part + p * nt;
  double v = 0.0;
  for (int t = threadIdx.x & 15; t < nt; t += 16) v += q[t];
  v += row_xor<8>(v);
  v += row_xor<4>(v);
  v += row_xor<2>(v);
  v += row_xor<1>(v);
  return a.y_mean + a.y_std * (a.c + v);
}

// V V^T of the 16 / mq whole batch elements in 16 consecutive rows: each wave
// takes a quarter of the columns (16 x 16 FP64 MFMA; the lanes' 16-byte loads
// cover 64 bytes of a row per step, eight steps in flight), the quarters are
// added through LDS, then one thread per (i, j) pair writes its output.  Rows
// past the group repeat the last one and are not read by any output.
__global__ __launch_bounds__(256) void post_cov_small_kernel(PostOutArgs a) {
  __shared__ double red[4][16][17];
  __shared__ double xr[16][PC_MAXD + 1];
  const int mq = a.rows.mq, d = a.d;
  const int per = 16 / mq * mq;  // rows per block
  const int64_t R = a.rows.batch * mq, r0 = (int64_t)blockIdx.x * per;
  const int nr = (int)min((int64_t)per, R - r0);
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6, l16 = lane & 15, g = lane >> 4;
  for (int i = threadIdx.x; i < nr * d; i += 256) xr[i / d][i % d] = a.xs[r0 * d + i];
  const double* v = a.V + (r0 + min(l16, nr - 1)) * a.n_pad + wv * (a.n_pad / 4) + 2 * g;
  const int steps = (int)(a.n_pad / 32);  // 8 columns each; a multiple of 4
  v4d acc0 = (v4d)(0.0), acc1 = (v4d)(0.0);
  for (int t0 = 0; t0 < steps; t0 += 8) {
    v2d x[8];
#pragma unroll
    for (int u = 0; u < 8; ++u)
      x[u] = t0 + u < steps ? *(const v2d*)(v + 8 * (t0 + u)) : (v2d)(0.0);
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      acc0 = __builtin_amdgcn_mfma_f64_16x16x4f64(x[u].x, x[u].x, acc0, 0, 0, 0);
      acc1 = __builtin_amdgcn_mfma_f64_16x16x4f64(x[u].y, x[u].y, acc1, 0, 0, 0);
    }
  }
#pragma unroll
  for (int q = 0; q < 4; ++q) red[wv][Mfma<double>::row(g, q)][l16] = acc0[q] + acc1[q];
  __syncthreads();
  const int i = threadIdx.x >> 4, j = threadIdx.x & 15;
  if (a.mean) {
    const double mu = post_mean16(a, r0 + min(i, nr - 1));
    if (j == 0 && i < nr) a.mean[r0 + i] = mu;
  }
  if (i >= nr || j >= nr || i / mq != j / mq || !(a.covar || a.var)) return;
  double r2 = 0.0;
  for (int t = 0; t < d; ++t) {
    const double df = xr[i][t] - xr[j][t];
    r2 = fma(df, df, r2);
  }
  const double vv = (red[0][i][j] + red[1][i][j]) + (red[2][i][j] + red[3][i][j]);
  const double o = a.y_std * a.y_std * (kern_any(a.kind, r2, a.s) - vv);
  if (a.covar) a.covar[(r0 + i) * mq + j % mq] = o;
  if (a.var && i == j) a.var[r0 + i] = o;
}

// Lower 128 x 64 tile (tm, tn) of one batch element's mq_pad x mq_pad products,
// enumerated row by row (tn <= 2 tm + 1); the symmetric half is written from the
// same values.  Forming both halves, with the outputs copied out of the padded
// blocks by a kernel of their own, took 200 us at mq = 1500 and n = 1000.
template <int KIND>
__global__ __launch_bounds__(256, 2) void post_cov_joint_kernel(PostOutArgs a) {
  __shared__ __attribute__((aligned(1024)))
  unsigned char lds[DCfg<64>::STAGES * DCfg<64>::STAGE];
  const int mq = a.rows.mq, mp = a.rows.mq_pad, d = a.d;
  const int64_t bi = blockIdx.y;
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  const int wy = wv >> 1, wx = wv & 1, l16 = lane & 15, gq = lane >> 4;
  int tm = 0;
  while ((tm + 1) * (tm + 2) <= (int)blockIdx.x) ++tm;
  const int tn = (int)blockIdx.x - tm * (tm + 1);
  if (tn * 64 >= mp) return;  // (uniform) the last tile row may hold 64 rows only
  const double* V = a.V + bi * mp * a.n_pad;
  v4d acc[4][2];
  d_mainloop<64, false, false>(V, a.n_pad, V, a.n_pad, tm * D_BM, tn * 64, mp, mp, 0,
                               (int)a.n_pad, lds, acc);
  // the ring is free: the tile's rows and columns, in coordinate chunks of 16
  constexpr int DC = 16;
  double* xr = (double*)lds;           // 128 x 17
  double* xc = xr + D_BM * (DC + 1);   // 64 x 17
  const double* xs = a.xs + bi * mp * d;
  double r2[4][2][4];
#pragma unroll
  for (int mi = 0; mi < 4; ++mi)
#pragma unroll
    for (int ni = 0; ni < 2; ++ni)
#pragma unroll
      for (int q = 0; q < 4; ++q) r2[mi][ni][q] = 0.0;
  for (int j0 = 0; j0 < d; j0 += DC) {
    if (j0) __syncthreads();
    for (int e = threadIdx.x; e < (D_BM + 64) * DC; e += 256) {
      const int r = e / DC, j = j0 + e % DC;
      const int p = r < D_BM ? tm * D_BM + r : tn * 64 + r - D_BM;
      xr[r * (DC + 1) + e % DC] = (j < d && p < mq) ? xs[(int64_t)p * d + j] : 0.0;
    }
    __syncthreads();
    const int je = min(DC, d - j0);
    for (int j = 0; j < je; ++j) {
      double cv[2];
#pragma unroll
      for (int ni = 0; ni < 2; ++ni) cv[ni] = xc[(wx * 32 + ni * 16 + l16) * (DC + 1) + j];
#pragma unroll
      for (int mi = 0; mi < 4; ++mi)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const double rv = xr[(wy * 64 + mi * 16 + Mfma<double>::row(gq, q)) * (DC + 1) + j];
#pragma unroll
          for (int ni = 0; ni < 2; ++ni) {
            const double df = rv - cv[ni];
            r2[mi][ni][q] = fma(df, df, r2[mi][ni][q]);
          }
        }
    }
  }
  const double ys2 = a.y_std * a.y_std;
#pragma unroll
  for (int mi = 0; mi < 4; ++mi)
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int row = tm * D_BM + wy * 64 + mi * 16 + Mfma<double>::row(gq, q);
#pragma unroll
      for (int ni = 0; ni < 2; ++ni) {
        const int col = tn * 64 + wx * 32 + ni * 16 + l16;
        if (row >= mq || col > row) continue;
        const double o = ys2 * (kern_value_k<KIND>(r2[mi][ni][q], a.s) - acc[mi][ni][q]);
        if (a.covar) {
          a.covar[(bi * mq + row) * mq + col] = o;
          a.covar[(bi * mq + col) * mq + row] = o;
        }
        if (a.var && row == col) a.var[bi * mq + row] = o;
      }
    }
  if (a.mean && tn == 0)
    for (int r = threadIdx.x >> 4; r < D_BM; r += 16) {
      const int row = tm * D_BM + r;
      if (row >= mq) break;  // uniform over the 16 lanes of a row
      const double mu = post_mean16(a, bi * mp + row);
      if ((threadIdx.x & 15) == 0) a.mean[bi * mq + row] = mu;
    }
}

// The same from 32 x 32 lower tiles (gemm_w_body.h), for outputs of too few 128 x 64
// tiles to fill the chip: at mq = 1500, n = 1000 those are 156 tiles of which each
// runs 2048 matrix products a wave, 101 us; the 1176 small ones take 66 us.  Both
// halves are written in rows of 256 bytes from the tile in LDS.
template <int KIND>
__global__ __launch_bounds__(256, 2) void post_cov_tiles_kernel(PostOutArgs a) {
  constexpr int T = 32;
  __shared__ __attribute__((aligned(1024))) unsigned char lds[w_lds<2, 2, 4, 16, 2>()];
  static_assert(4 * T * T * 8 + 2 * T * (PC_MAXD + 1) * 8 <= w_lds<2, 2, 4, 16, 2>(),
                "the coordinates follow the partial tiles");
  const int mq = a.rows.mq, mp = a.rows.mq_pad, d = a.d;
  const int64_t bi = blockIdx.y;
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6, l16 = lane & 15, gq = lane >> 4;
  int ti, tj;
  decode_tile((int)blockIdx.x, BTA_GEMM_C_LOWER, mp / T, mp / T, ti, tj);
  const double* V = a.V + bi * mp * a.n_pad;
  const double* xs = a.xs + bi * mp * d;
  // the tile's row and column points, on their way during the products
  double xv[2 * T * PC_MAXD / 256];
#pragma unroll
  for (int u = 0; u < 2 * T * PC_MAXD / 256; ++u) {
    const int e = tid + 256 * u;
    xv[u] = 0.0;
    if (e < 2 * T * d) {
      const int r = e / d, p = r < T ? ti * T + r : tj * T + r - T;
      if (p < mq) xv[u] = xs[(int64_t)p * d + e % d];
    }
  }
  w_partials<2, 2, 4, 16, 2, false>(V, a.n_pad, V, a.n_pad, ti * T, tj * T, 0, (int)a.n_pad, lds);
  const double* red = (const double*)lds;
  double* xr = (double*)lds + 4 * T * T;  // 64 x (PC_MAXD + 1), rows then columns
#pragma unroll
  for (int u = 0; u < 2 * T * PC_MAXD / 256; ++u) {
    const int e = tid + 256 * u;
    if (e < 2 * T * d) xr[e / d * (PC_MAXD + 1) + e % d] = xv[u];
  }
  // wave wv finishes fragment (wv / 2, wv % 2)
  const int rl = 16 * (wv >> 1), cl = 16 * (wv & 1) + l16;
  double o[4], r2[4] = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
  for (int q = 0; q < 4; ++q) o[q] = w_sum<2, 2, 4>(red, wv, q, lane);
  __syncthreads();
  for (int j = 0; j < d; ++j) {
    const double c = xr[(T + cl) * (PC_MAXD + 1) + j];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const double df = xr[(rl + Mfma<double>::row(gq, q)) * (PC_MAXD + 1) + j] - c;
      r2[q] = fma(df, df, r2[q]);
    }
  }
  double* ot = (double*)lds;  // 32 x 33 (the partial tiles are read)
  const double ys2 = a.y_std * a.y_std;
#pragma unroll
  for (int q = 0; q < 4; ++q)
    ot[(rl + Mfma<double>::row(gq, q)) * (T + 1) + cl] =
        ys2 * (kern_value_k<KIND>(r2[q], a.s) - o[q]);
  __syncthreads();
  for (int e = tid; e < T * T; e += 256) {
    const int r = e / T, c = e % T;
    const int row = ti * T + r, col = tj * T + c;
    const double lo = ot[r * (T + 1) + c], up = ot[c * (T + 1) + r];
    if (a.covar) {
      if (row < mq && col < mq) a.covar[(bi * mq + row) * mq + col] = ti > tj || c <= r ? lo : up;
      if (ti > tj && ti * T + c < mq)  // (tj's rows are all in use then)
        a.covar[(bi * mq + tj * T + r) * mq + ti * T + c] = up;
    }
    if (a.var && row == col && row < mq) a.var[bi * mq + row] = lo;
  }
  if (a.mean && tj == 0)
    for (int r = tid >> 4; r < T; r += 16) {
      const int row = ti * T + r;
      if (row >= mq) break;  // uniform over the 16 lanes of a row
      const double mu = post_mean16(a, bi * mp + row);
      if ((tid & 15) == 0) a.mean[bi * mq + row] = mu;
    }
}

// Row layout of a call: mq_pad and the total of padded rows.
struct PostLayout {
  int mq_pad;
  int64_t R_pad;
  PostLayout(int64_t batch, int mq) {
    if (mq <= POST_SMALL_MQ) {
      mq_pad = mq;
      R_pad = round_up(batch * mq, 128);
    } else {
      mq_pad = (int)round_up(mq, 64);
      R_pad = batch * mq_pad;
    }
  }
  // rows the products have to form
  int64_t used(int64_t batch, int mq) const { return mq_pad == mq ? batch * mq : R_pad; }
};

struct PostWs {
  PostLayout lay;
  size_t xs, kx, vt, part, total;
  PostWs(const bta_gp_model* m, int64_t batch, int mq) : lay(batch, mq) {
    WsPlan p;
    xs = p.take((size_t)lay.R_pad * m->d * 8);
    kx = p.take((size_t)lay.R_pad * m->n_pad * 8);
    vt = p.take((size_t)lay.R_pad * m->n_pad * 8);
    part = p.take((size_t)lay.R_pad * (m->n_pad / 64) * 8);
    total = p.off;
  }
};

// What the adjoint takes over from the moments of the same call: xs and V.
struct PostKeep {
  size_t xs, vt, total;
  PostKeep(const bta_gp_model* m, const PostLayout& lay) {
    WsPlan p;
    xs = p.take((size_t)lay.R_pad * m->d * 8);
    vt = p.take((size_t)lay.R_pad * m->n_pad * 8);
    total = p.off;
  }
};

static int post_check(const char* what, const bta_gp_model* m, int64_t batch, int mq) {
  if (m->d < 1 || m->d > PC_MAXD || m->n < 1 || m->n_pad < m->n || m->n_pad % 128) {
    set_error("%s: bad sizes (d=%d n=%ld n_pad=%ld)", what, m->d, (long)m->n, (long)m->n_pad);
    return BTA_ERR_INVALID;
  }
  if (batch * round_up(mq, 64) > (int64_t)8 * 65535) {
    set_error("%s: too many rows", what);
    return BTA_ERR_UNSUPPORTED;
  }
  return BTA_OK;
}

// xs, K_x (and the partials of K_x alpha) of the batch's rows
static int post_rows(const bta_gp_model* m, const double* X, int64_t batch, int mq,
                     const PostLayout& lay, double* xs, double* kx, double* part, hipStream_t s) {
  PostCovarArgs c;
  c.X = X;
  c.rows = PostRows{batch, mq, lay.mq_pad};
  c.center = m->center;
  c.ls = m->lengthscale;
  c.T = m->train_xs;
  c.alpha = m->alpha;
  c.xs = xs;
  c.K = kx;
  c.part = part;
  c.n = m->n;
  c.n_pad = m->n_pad;
  c.d = m->d;
  c.s = m->outputscale;
  return post_covar(c, m->kind, lay.R_pad, s);
}

int gp_posterior(const bta_gp_model* m, const double* X, int64_t batch, int mq, double* mean,
                 double* covar_out, double* var, void* keep, void* ws, size_t ws_bytes,
                 hipStream_t s) {
  if (!m || !X || batch < 1 || mq < 1 || !m->linv || !m->alpha || batch > 65535) {
    set_error("gp_posterior: invalid arguments");
    return BTA_ERR_INVALID;
  }
  int rc = post_check("gp_posterior", m, batch, mq);
  if (rc) return rc;
  const PostWs w(m, batch, mq);
  if (!ws || ws_bytes < w.total) {
    set_error("gp_posterior: workspace too small");
    return BTA_ERR_WORKSPACE;
  }
  char* base = (char*)ws;
  double* xs = (double*)(base + w.xs);
  double* kx = (double*)(base + w.kx);
  double* vt = (double*)(base + w.vt);
  double* part = (double*)(base + w.part);
  if (keep) {
    const PostKeep k(m, w.lay);
    xs = (double*)((char*)keep + k.xs);
    vt = (double*)((char*)keep + k.vt);
  }
  const int64_t np = m->n_pad;
  rc = post_rows(m, X, batch, mq, w.lay, xs, kx, part, s);
  if (rc) return rc;
  rc = gemm_rows(BTA_GEMM_B_LOWER, w.lay.used(batch, mq), w.lay.R_pad, np, kx, m->linv, vt, s);
  if (rc) return rc;
  PostOutArgs o;
  o.V = vt;
  o.xs = xs;
  o.part = part;
  o.rows = PostRows{batch, mq, w.lay.mq_pad};
  o.n_pad = np;
  o.d = m->d;
  o.kind = m->kind;
  o.s = m->outputscale;
  o.y_mean = m->y_mean;
  o.y_std = m->y_std;
  o.c = m->mean_constant;
  o.mean = mean;
  o.covar = covar_out;
  o.var = var;
  if (mq <= POST_SMALL_MQ) {
    const int per = 16 / mq * mq;
    hipLaunchKernelGGL(post_cov_small_kernel, dim3((unsigned)((batch * mq + per - 1) / per)),
                       dim3(256), 0, s, o);
  } else {
    const int MT = (w.lay.mq_pad + D_BM - 1) / D_BM, TT = w.lay.mq_pad / 32;
    const bool m52 = m->kind == BTA_KERNEL_MATERN52;
    // small tiles below 1.5 large ones per CU, as for the products of gemm_w.hip
    const bool small = 2 * (int64_t)MT * (MT + 1) * batch < 3 * (int64_t)num_cus();
    const dim3 g((unsigned)(small ? TT * (TT + 1) / 2 : MT * (MT + 1)), (unsigned)batch);
    if (small && m52)
      hipLaunchKernelGGL((post_cov_tiles_kernel<BTA_KERNEL_MATERN52>), g, dim3(256), 0, s, o);
    else if (small)
      hipLaunchKernelGGL((post_cov_tiles_kernel<BTA_KERNEL_RBF>), g, dim3(256), 0, s, o);
    else if (m52)
      hipLaunchKernelGGL((post_cov_joint_kernel<BTA_KERNEL_MATERN52>), g, dim3(256), 0, s, o);
    else
      hipLaunchKernelGGL((post_cov_joint_kernel<BTA_KERNEL_RBF>), g, dim3(256), 0, s, o);
  }
  BTA_LAUNCH_CHECK("post_cov kernel");
  return BTA_OK;
}

// ---------------------------------------------------------------------------
// Adjoint of the posterior: dX from d mean and d covar.
//   dK_x   = y_std dmean alpha^T - y_std^2 (dC + dC^T) U,   U = V L^-1 = K_x K^-1
//   dK_xx  = y_std^2 dC  (the prior covariance among the batch's own points)
//   dX     = through dk/dX of both, divided by the lengthscale
// ---------------------------------------------------------------------------
struct PostGradArgs {
  const double *xs, *T, *alpha, *U;  // U: R_pad x n_pad; with G given, G = -S U
  const double *dmean, *dcov;        // either may be null
  PostRows rows;
  double* part;  // splits x R x d
  int64_t R_pad, n, n_pad;
  int d, splits;
  double s, y_std;
};

// S_b[i][j] = y_std^2 (dC_b + dC_b^T) zero-padded to mq_pad x mq_pad, for the
// products with whole padded elements (mq > POST_SMALL_MQ)
__global__ void post_bwd_prep_kernel(const double* dcov, int mq, int mq_pad, double y_std,
                                     double* S) {
  const int64_t bi = blockIdx.y;
  for (int e = blockIdx.x * blockDim.x + threadIdx.x; e < mq_pad * mq_pad;
       e += gridDim.x * blockDim.x) {
    const int i = e / mq_pad, j = e % mq_pad;
    double v = 0.0;
    if (i < mq && j < mq)
      v = y_std * y_std * (dcov[(bi * mq + i) * mq + j] + dcov[(bi * mq + j) * mq + i]);
    S[bi * mq_pad * mq_pad + e] = v;
  }
}

// RB rows per block, one column per thread and pass, columns c = 256 (split +
// k splits) + thread.  MIX: the block's rows read U of their own batch elements
// and mix it with S from LDS (at most 2 RB - 1 elements meet RB rows; each U value
// is read once for the rows of its element); otherwise U holds -S U already.
// With RB x MD accumulators and the point's MD coordinates in registers the
// kernel is bound by its FP64 VALU work (3 d + ~45 instructions an element).
template <int RB, int MD, int KIND, bool MIX>
__global__ __launch_bounds__(256) void post_grad_kernel(PostGradArgs a) {
  __shared__ double xr[RB * MD];
  __shared__ double Sr[MIX ? RB * POST_SMALL_MQ : 1];
  __shared__ double dm[RB];
  __shared__ double red[4][RB * MD];
  const int d = a.d, mq = a.rows.mq;
  const int64_t r0 = (int64_t)blockIdx.x * RB;
  for (int i = threadIdx.x; i < RB * MD; i += 256) {
    const int64_t p = r0 + i / MD;
    xr[i] = (i % MD < d && p < a.R_pad) ? a.xs[p * d + i % MD] : 0.0;
  }
  if (MIX)
    for (int i = threadIdx.x; i < RB * mq; i += 256) {
      int64_t bi;
      int r;
      const int j = i % mq;
      const bool ok = a.dcov && a.rows.at(r0 + i / mq, bi, r);
      Sr[(i / mq) * POST_SMALL_MQ + j] =
          ok ? a.y_std * a.y_std *
                   (a.dcov[(bi * mq + r) * mq + j] + a.dcov[(bi * mq + j) * mq + r])
             : 0.0;
    }
  if (threadIdx.x < RB) {
    int64_t bi;
    int r;
    const bool ok = a.dmean && a.rows.at(r0 + threadIdx.x, bi, r);
    dm[threadIdx.x] = ok ? a.y_std * a.dmean[bi * mq + r] : 0.0;
  }
  __syncthreads();
  double acc[RB][MD];
#pragma unroll
  for (int q = 0; q < RB; ++q)
#pragma unroll
    for (int j = 0; j < MD; ++j) acc[q][j] = 0.0;
  for (int64_t c0 = (int64_t)blockIdx.y * PG_COLS; c0 < a.n; c0 += (int64_t)a.splits * PG_COLS) {
    const int64_t c = c0 + threadIdx.x;
    if (c >= a.n) break;
    double t[MD];
#pragma unroll
    for (int j = 0; j < MD; ++j) t[j] = j < d ? a.T[c * d + j] : 0.0;
    const double al = a.dmean ? a.alpha[c] : 0.0;
    double gv[RB];
#pragma unroll
    for (int q = 0; q < RB; ++q) gv[q] = dm[q] * al;
    if (a.dcov) {
      if (MIX) {
        // rows r0 .. r0 + RB - 1 lie in elements b0 .. b1
        const int64_t b0 = r0 / mq;
        const int64_t b1 = min((r0 + RB - 1) / mq, a.rows.batch - 1);
        for (int64_t b = b0; b <= b1; ++b) {
          const double* u = a.U + b * mq * a.n_pad + c;
          const int off = (int)(b * mq - r0);  // rows off .. off + mq - 1 of the block
          for (int j = 0; j < mq; ++j) {
            const double uv = u[j * a.n_pad];
#pragma unroll
            for (int q = 0; q < RB; ++q)
              if (q >= off && q < off + mq) gv[q] = fma(-Sr[q * POST_SMALL_MQ + j], uv, gv[q]);
          }
        }
      } else {
#pragma unroll
        for (int q = 0; q < RB; ++q)
          if (r0 + q < a.R_pad) gv[q] += a.U[(r0 + q) * a.n_pad + c];
      }
    }
#pragma unroll
    for (int q = 0; q < RB; ++q) {
      double r2 = 0.0;
#pragma unroll
      for (int j = 0; j < MD; ++j) {
        const double df = xr[q * MD + j] - t[j];
        r2 = fma(df, df, r2);
      }
      const double w = -gv[q] * kern_grad_factor_k<KIND>(r2, a.s);
#pragma unroll
      for (int j = 0; j < MD; ++j) acc[q][j] = fma(w, xr[q * MD + j] - t[j], acc[q][j]);
    }
  }
  const int wv = threadIdx.x >> 6;
#pragma unroll
  for (int q = 0; q < RB; ++q) {
    int e;
    const double v = wave_sum_spread<MD>(acc[q], &e);
    if (e >= 0) red[wv][q * MD + e] = v;
  }
  __syncthreads();
  const int64_t R = a.rows.batch * mq;
  for (int i = threadIdx.x; i < RB * d; i += 256) {
    const int q = i / d, j = i % d;
    int64_t bi;
    int r;
    if (!a.rows.at(r0 + q, bi, r)) continue;
    const int e = q * MD + j;
    a.part[((int64_t)blockIdx.y * R + bi * mq + r) * d + j] =
        (red[0][e] + red[1][e]) + (red[2][e] + red[3][e]);
  }
}

// dX[r][j] = (sum over the splits + sum_i2 S_b[i][i2] dk(xs_i, xs_i2)/dxs_i[j]) / l_j,
// one 16-lane group per row: the lanes share the other points i2 of the element.
template <int KIND>
__global__ __launch_bounds__(256) void post_grad_finish_kernel(PostGradArgs a,
                                                               const double* __restrict__ ls,
                                                               double* __restrict__ dX) {
  const int mq = a.rows.mq, mp = a.rows.mq_pad, d = a.d, sub = threadIdx.x & 15;
  const int64_t R = a.rows.batch * mq;
  const int64_t row = (int64_t)blockIdx.x * 16 + (threadIdx.x >> 4);
  if (row >= R) return;  // uniform over the row's lanes
  const int64_t bi = row / mq;
  const int i = (int)(row % mq);
  const double* xb = a.xs + bi * mp * d;
  double acc[PC_MAXD];
#pragma unroll
  for (int j = 0; j < PC_MAXD; ++j) acc[j] = 0.0;
  if (a.dcov)
    for (int i2 = sub; i2 < mq; i2 += 16) {
      if (i2 == i) continue;
      const double sv = a.y_std * a.y_std *
                        (a.dcov[(bi * mq + i) * mq + i2] + a.dcov[(bi * mq + i2) * mq + i]);
      if (sv == 0.0) continue;
      double r2 = 0.0, df[PC_MAXD];
#pragma unroll
      for (int j = 0; j < PC_MAXD; ++j) {
        df[j] = j < d ? xb[i * d + j] - xb[i2 * d + j] : 0.0;
        r2 = fma(df[j], df[j], r2);
      }
      const double w = -sv * kern_grad_factor_k<KIND>(r2, a.s);
#pragma unroll
      for (int j = 0; j < PC_MAXD; ++j) acc[j] = fma(w, df[j], acc[j]);
    }
#pragma unroll
  for (int j = 0; j < PC_MAXD; ++j) {
    if (j >= d) break;
    double v = acc[j];
    v += row_xor<8>(v);
    v += row_xor<4>(v);
    v += row_xor<2>(v);
    v += row_xor<1>(v);
    if (sub == (j & 15)) {
      for (int sp = 0; sp < a.splits; ++sp) v += a.part[((int64_t)sp * R + row) * d + j];
      dX[row * d + j] = v / ls[j];
    }
  }
}

constexpr int POST_MAX_SPLITS = 16;

// Column shares of post_grad_kernel: enough blocks for two per CU when the rows
// alone do not give them, at most one share per 256 columns.
static int post_grad_splits(int64_t row_blocks, int64_t n) {
  const int64_t want = (2 * (int64_t)num_cus() + row_blocks - 1) / row_blocks;
  return (int)std::max<int64_t>(
      1, std::min<int64_t>({want, (n + PG_COLS - 1) / PG_COLS, POST_MAX_SPLITS}));
}

struct PostBwdWs {
  PostLayout lay;
  size_t xs, kx, vt, S, part, total;
  PostBwdWs(const bta_gp_model* m, int64_t batch, int mq) : lay(batch, mq) {
    WsPlan p;
    xs = p.take((size_t)lay.R_pad * m->d * 8);
    kx = p.take((size_t)lay.R_pad * m->n_pad * 8);
    vt = p.take((size_t)lay.R_pad * m->n_pad * 8);
    S = p.take(mq > POST_SMALL_MQ ? (size_t)batch * lay.mq_pad * lay.mq_pad * 8 : 0);
    part = p.take((size_t)POST_MAX_SPLITS * batch * mq * m->d * 8);
    total = p.off;
  }
};

template <int RB, int MD, int KIND>
static void post_grad_mode(const PostGradArgs& a, bool mix, dim3 g, hipStream_t s) {
  if (mix)
    hipLaunchKernelGGL((post_grad_kernel<RB, MD, KIND, true>), g, dim3(256), 0, s, a);
  else
    hipLaunchKernelGGL((post_grad_kernel<RB, MD, KIND, false>), g, dim3(256), 0, s, a);
}

template <int RB, int MD>
static void post_grad_kind(PostGradArgs& a, int kind, bool mix, hipStream_t s) {
  const int64_t nb = (a.R_pad + RB - 1) / RB;
  a.splits = post_grad_splits(nb, a.n);
  const dim3 g((unsigned)nb, (unsigned)a.splits);
  if (kind == BTA_KERNEL_MATERN52)
    post_grad_mode<RB, MD, BTA_KERNEL_MATERN52>(a, mix, g, s);
  else
    post_grad_mode<RB, MD, BTA_KERNEL_RBF>(a, mix, g, s);
}

// keep: null, or the xs and V of the moments' call (X is then not read)
int gp_posterior_backward(const bta_gp_model* m, const double* X, int64_t batch, int mq,
                          const double* dmean, const double* dcov, double* dX, const void* keep,
                          void* ws, size_t ws_bytes, hipStream_t s) {
  if (!m || (!X && !keep) || !dX || batch < 1 || mq < 1 || !m->linv || !m->alpha || batch > 65535 ||
      (!dmean && !dcov)) {
    set_error("gp_posterior_backward: invalid arguments");
    return BTA_ERR_INVALID;
  }
  int rc = post_check("gp_posterior_backward", m, batch, mq);
  if (rc) return rc;
  const PostBwdWs w(m, batch, mq);
  if (!ws || ws_bytes < w.total) {
    set_error("gp_posterior_backward: workspace too small");
    return BTA_ERR_WORKSPACE;
  }
  char* base = (char*)ws;
  double* xs = (double*)(base + w.xs);
  double* kx = (double*)(base + w.kx);
  double* vt = (double*)(base + w.vt);
  double* S = (double*)(base + w.S);
  const int64_t np = m->n_pad, mp = w.lay.mq_pad, R_pad = w.lay.R_pad;
  const bool mix = mq <= POST_SMALL_MQ;
  const double* V = vt;
  if (keep) {
    const PostKeep k(m, w.lay);
    xs = (double*)((char*)keep + k.xs);
    V = (const double*)((const char*)keep + k.vt);
  } else {
    rc = post_rows(m, X, batch, mq, w.lay, xs, kx, nullptr, s);
    if (rc) return rc;
  }
  PostGradArgs a;
  a.U = nullptr;
  if (dcov) {
    // V = K_x L^-T into vt (unless it was kept), then U = V L^-1 into kx
    const int64_t R = w.lay.used(batch, mq);
    if (!keep) {
      rc = gemm_rows(BTA_GEMM_B_LOWER, R, R_pad, np, kx, m->linv, vt, s);
      if (rc) return rc;
    }
    rc = gemm_rows(BTA_GEMM_B_KN | BTA_GEMM_B_UPPER, R, R_pad, np, V, m->linv, kx, s);
    if (rc) return rc;
    a.U = kx;
    if (!mix) {
      // -S U per padded batch element, into vt
      const dim3 g((unsigned)std::min<int64_t>(1024, (mp * mp + 255) / 256), (unsigned)batch);
      hipLaunchKernelGGL(post_bwd_prep_kernel, g, dim3(256), 0, s, dcov, mq, w.lay.mq_pad,
                         m->y_std, S);
      BTA_LAUNCH_CHECK("post_bwd_prep_kernel");
      rc = gemm(BTA_GEMM_B_KN, mp, np, mp, -1.0, S, mp, kx, np, 0.0, nullptr, 0, vt, np, s,
                (int)batch, mp * mp, mp * np, 0, mp * np);
      if (rc) return rc;
      a.U = vt;
    }
  }
  a.xs = xs;
  a.T = m->train_xs;
  a.alpha = m->alpha;
  a.dmean = dmean;
  a.dcov = dcov;
  a.rows = PostRows{batch, mq, w.lay.mq_pad};
  a.part = (double*)(base + w.part);
  a.R_pad = R_pad;
  a.n = m->n;
  a.n_pad = np;
  a.d = m->d;
  a.s = m->outputscale;
  a.y_std = m->y_std;
  switch ((m->d + 3) / 4) {
    case 1: post_grad_kind<4, 4>(a, m->kind, mix, s); break;
    case 2: post_grad_kind<4, 8>(a, m->kind, mix, s); break;
    case 3: post_grad_kind<4, 12>(a, m->kind, mix, s); break;
    case 4: post_grad_kind<4, 16>(a, m->kind, mix, s); break;
    case 5: post_grad_kind<2, 20>(a, m->kind, mix, s); break;
    case 6: post_grad_kind<2, 24>(a, m->kind, mix, s); break;
    case 7: post_grad_kind<2, 28>(a, m->kind, mix, s); break;
    default: post_grad_kind<2, 32>(a, m->kind, mix, s); break;
  }
  BTA_LAUNCH_CHECK("post_grad_kernel");
  const dim3 gf((unsigned)((batch * mq + 15) / 16));
  if (m->kind == BTA_KERNEL_MATERN52)
    hipLaunchKernelGGL((post_grad_finish_kernel<BTA_KERNEL_MATERN52>), gf, dim3(256), 0, s, a,
                       m->lengthscale, dX);
  else
    hipLaunchKernelGGL((post_grad_finish_kernel<BTA_KERNEL_RBF>), gf, dim3(256), 0, s, a,
                       m->lengthscale, dX);
  BTA_LAUNCH_CHECK("post_grad_finish_kernel");
  return BTA_OK;
}

}  // namespace bta

extern "C" size_t bta_gp_posterior_workspace_size(const bta_gp_model* m, int64_t batch,
                                                  int32_t mq) {
  if (!m || batch < 1 || mq < 1) return 0;
  return bta::PostWs(m, batch, mq).total;
}

extern "C" int bta_gp_posterior(const bta_gp_model* m, const double* X, int64_t batch,
                                int32_t mq, double* mean, double* covar, double* var, void* ws,
                                size_t ws_bytes, bta_stream_t stream) {
  return bta::gp_posterior(m, X, batch, mq, mean, covar, var, nullptr, ws, ws_bytes,
                           (hipStream_t)stream);
}

extern "C" size_t bta_gp_posterior_keep_size(const bta_gp_model* m, int64_t batch, int32_t mq) {
  if (!m || batch < 1 || mq < 1) return 0;
  return bta::PostKeep(m, bta::PostLayout(batch, mq)).total;
}

extern "C" int bta_gp_posterior_keep(const bta_gp_model* m, const double* X, int64_t batch,
                                     int32_t mq, double* mean, double* covar, double* var,
                                     void* keep, void* ws, size_t ws_bytes,
                                     bta_stream_t stream) {
  if (!keep) {
    bta::set_error("gp_posterior_keep: null pointer");
    return BTA_ERR_INVALID;
  }
  return bta::gp_posterior(m, X, batch, mq, mean, covar, var, keep, ws, ws_bytes,
                           (hipStream_t)stream);
}

extern "C" int bta_gp_posterior_backward_kept(const bta_gp_model* m, int64_t batch, int32_t mq,
                                              const double* dmean, const double* dcov,
                                              double* dX, const void* keep, void* ws,
                                              size_t ws_bytes, bta_stream_t stream) {
  if (!keep) {
    bta::set_error("gp_posterior_backward_kept: null pointer");
    return BTA_ERR_INVALID;
  }
  return bta::gp_posterior_backward(m, nullptr, batch, mq, dmean, dcov, dX, keep, ws, ws_bytes,
                                    (hipStream_t)stream);
}

extern "C" size_t bta_gp_posterior_backward_workspace_size(const bta_gp_model* m,
                                                          int64_t batch, int32_t mq) {
  if (!m || batch < 1 || mq < 1) return 0;
  return bta::PostBwdWs(m, batch, mq).total;
}

extern "C" int bta_gp_posterior_backward(const bta_gp_model* m, const double* X, int64_t batch,
                                         int32_t mq, const double* dmean, const double* dcov,
                                         double* dX, void* ws, size_t ws_bytes,
                                         bta_stream_t stream) {
  if (!X) {
    bta::set_error("gp_posterior_backward: invalid arguments");
    return BTA_ERR_INVALID;
  }
  return bta::gp_posterior_backward(m, X, batch, mq, dmean, dcov, dX, nullptr, ws, ws_bytes,
                                    (hipStream_t)stream);
}
