// Split-FP16 GEMM on pre-split operands ("h2"):
//   C = alpha * (A_hi + A_lo/2^11)(B_hi + B_lo/2^11)^T / (a_scale a_row_scale[r] b_scale)
// with the lo x lo term dropped (2^-22 relative).  A plane pair holds
// hi = fp16(x) and lo = fp16(2^11 (x - hi)): the lo plane stays in FP16's normal
// range for small x, so every entry keeps ~22 significant bits.  A (M x K) and
// B (N x K) are two FP16 planes each, K-contiguous, written by their producers
// (the covariance kernel, this GEMM's own split epilogue, the factor set-up),
// so the main loop is data movement plus three v_mfma_f32_16x16x32_f16 per
// fragment pair.  hi x hi and the two cross products accumulate in separate
// FP32 sets (the cross set weighted by 2^-11 when combined), either over the
// whole K range (default) or in FP32 segments of k_segment added into FP64
// sums.  With the lo planes in range, the operand representation dominates
// the error: FP32 accumulation over K = 2048 leaves V V^T as accurate as FP64
// segment sums do, so the default path keeps no FP64 accumulators and runs
// two workgroups (two waves per SIMD) on each CU.
//
// Operands move global -> LDS with direct LDS loads (global_load_lds_dwordx4: no
// registers, no ds_write) through a ring of three LDS stages with two chunks of 32
// K in flight; one barrier per chunk.  A stage row is 128 bytes, a row's chunk of
// both planes, with the eight 16-byte pieces in slots XOR-ed by the row: every
// ds_read_b128 is free of bank conflicts (SQ_LDS_BANK_CONFLICT 0; 64-byte rows
// per plane had two-way conflicts, about 4 cycles a read).  The first third of a
// chunk's products starts once the lo plane of A and the hi plane of B are in
// registers.  The epilogue writes C in FP32 and, optionally, C's own hi/lo planes
// (scaled by c_scale) for a following split GEMM.
//
// Four tiles, which give bit-identical results (us per triangular product M x N x
// N; the 128 x 64 and 128 x 128 tiles with 64-byte rows that they replace in the
// last column; shapes of one line were measured in one run):
//                      64 x 64   128 x 64   128 x 128   128 x 256   before
//     512 x  2048         24         34          42          74         42
//     512 x  4096         48         62          79         136         79
//    2048 x  2048         54         37          44          74         44
//    4096 x  2048                    70          59          80         71
//    2048 x  4096                   128         107         144        125
//    4096 x  4096        315        248         203         184        200
//    8192 x 16384      11600       9500                    6300       9500
// 64 x 64 (three workgroups per CU) has the shortest chunk, 0.3 us against 0.5,
// which is what counts while each CU has one tile or less; 128 x 256 with eight
// waves of 64 x 64 moves half the bytes per product and runs large products at the
// rate of a plain FP16 matrix product (1047 TFLOP/s in the last line, 970 inside a whole
// step of that size; plain 1030-1090), 128 x 128 with sixteen waves
// of 32 x 32 fills the gap where 128 x 256 gives a CU one tile only.  128 x 64 lies
// between, and is the tile of the launches that share CUs with other work.
// Triangular K ranges follow gemm_kernel; for 128 x 64 a cost model picks the
// worker count, and workers pair heavy with light tiles on each CU.
#include "bta_common.h"
#include "gemm.h"
#include "gemm_d.h"
#include "gemm_tile.h"
#include "kernels.h"
#include "gemm_h2_body.h"

#include <algorithm>
#include <cstdlib>
#include <map>
#include <mutex>
#include <tuple>
#include <vector>

namespace bta {

template <bool ACC64>
__global__ __launch_bounds__(256, (ACC64 ? 1 : 2)) void gemm_h2_kernel(H2Args g) {
  __shared__ __attribute__((aligned(1024)))
  unsigned char lds[H2Mid::STAGES * H2Mid::STAGE];
  gemm_h2_body<ACC64>(g, blockIdx.x, gridDim.x, lds);
}

// One workgroup per tile, longest first.  64 x 64 tiles: odd rounds of one
// workgroup per CU run backwards, so the workgroups sharing a CU hold long and
// short tiles (the larger tiles have a CU each and keep the order: 128 x 256, 196
// against 230 us at 4096 x 4096 with reversed rounds).
template <typename CFG, bool REV>
__global__ __launch_bounds__(64 * CFG::NW, (CFG::NW == 4 ? 3 : CFG::NW / 4)) void gemm_h2_tiles_kernel(
    H2Args g, int ncu) {
  __shared__ __attribute__((aligned(1024))) unsigned char lds[CFG::STAGES * CFG::STAGE];
  const int MT = g.M / CFG::TM, NT = (g.N + CFG::TN - 1) / CFG::TN, total = MT * NT;
  int t = blockIdx.x;
  if (REV) {
    const int rd = t / ncu;
    if (rd & 1) t = rd * ncu + min(ncu, total - rd * ncu) - 1 - (t - rd * ncu);
  }
  int tm, tn;
  decode_tile(t, g.flags, MT, NT, tm, tn);
  gemm_h2_tile(CFG(), g, tm, tn, lds);
}

// Cost model of the worker schedule: chunk counts per worker (plus a per-tile
// fixed cost); a CU's time is the sum over the workers it hosts, worker w on
// CU w % ncu.
static double h2_cost(const H2Args& g, int W) {
  constexpr int BN = H2Mid::TN;
  const int MT = g.M / H2_BM, NT = g.N / BN, total = MT * NT;
  const int ncu = num_cus();
  std::vector<double> cu(ncu, 0.0);
  const double per_chunk = 0.55;  // MFMA + LDS time of one K chunk
  for (int w = 0; w < W; ++w) {
    double load = 0.0;
    for (int j = 0; j * W < total; ++j) {
      const int t = h2_tile_of(j, w, W);
      if (t >= total) continue;
      int tm, tn;
      decode_tile(t, g.flags, MT, NT, tm, tn);
      int kb = 0, ke = g.K;
      if (g.flags & BTA_GEMM_B_LOWER) ke = std::min(ke, (tn + 1) * BN);
      if (g.flags & BTA_GEMM_B_UPPER) kb = std::max(kb, tn * BN);
      load += per_chunk * (ke > kb ? (ke - kb) / H2_BK : 0) + 6.0;
    }
    cu[w % ncu] += load;
  }
  return *std::max_element(cu.begin(), cu.end());
}

// bn: tile width.  64 with xcd >= 1: 128 x 64 tiles dealt to `workers` workgroups;
// with xcd 0 one workgroup per tile, 64 x 64 tiles for 64, 128 x bn above.
struct H2Plan {
  int bn, workers, xcd;
  bool tuned;
};

// Worker groups for gemm_h2_body's strip dealing: one per XCD (workgroups go
// to the XCDs round-robin by id; 32 CUs per XCD), when the tile order is strip
// by strip (triangular B), the strips pair up evenly across the groups (a
// multiple of 2 G of them) and the worker count divides evenly.  Off unless
// BTA_H2_XCD=1 is set: it lets one L2 serve each L^-1 strip, but on the
// 2048 x 2048 x 2048 step products it measured no faster (50.7-52.6 us against
// 50.2-52.9 us per forward product, step 0.189-0.193 ms against 0.185-0.187 ms).
static int h2_xcd_allowed(const H2Args& g, int W) {
  const int G = num_cus() / 32;
  if (G < 2 || !(g.flags & (BTA_GEMM_B_LOWER | BTA_GEMM_B_UPPER)) || W % G ||
      (g.N / H2Mid::TN) % (2 * G))
    return 1;
  return G;
}

static int h2_xcd_groups(const H2Args& g, int W) {
  static const int on = [] {
    const char* e = getenv("BTA_H2_XCD");
    return e && e[0] == '1';
  }();
  return on ? h2_xcd_allowed(g, W) : 1;
}

static int h2_tiles(const H2Args& g, int tm, int tn) {
  return (int)((int64_t)(g.M / tm) * ((g.N + tn - 1) / tn));
}

// The plans per problem signature: filled by the cost model below on a shape's
// first call, or by the measured tuner (gemm_h2_set_plan).  Never destroyed (no
// exit-time destructor; see plan_gemm).
typedef std::tuple<int, int, int, int, int> H2Key;
static std::mutex& h2_mu() {
  static std::mutex& mu = *new std::mutex;
  return mu;
}
static std::map<H2Key, H2Plan>& h2_cache() {
  static auto& cache = *new std::map<H2Key, H2Plan>;
  return cache;
}

// 128 x 64 tiles with the cost model's worker count
static H2Plan h2_mid_plan(const H2Args& g, bool acc64) {
  const int ncu = num_cus();
  const int slots = acc64 ? ncu : 2 * ncu;  // resident workgroups
  H2Plan best{64, 1, 1, false};
  double bt = 1e300;
  const int total = h2_tiles(g, H2Mid::TM, H2Mid::TN);
  for (int c : {slots, slots / 2, 3 * slots / 8, slots / 4}) {
    const int W = std::max(1, std::min(c, total));
    const double t = h2_cost(g, W);
    if (t < bt) {
      bt = t;
      best = {64, W, h2_xcd_groups(g, W), false};
    }
  }
  return best;
}

// The tile by the number of tiles the chip would get (table at the top): 64 x 64
// while the 128 x 64 tiles leave every CU at most one, 128 x 256 from 1.5 of its
// own per CU (3072 x 4096: 158 us, 128 x 128 165, 128 x 64 162), 128 x 128 from 1.75
// of its own, 128 x 64 between.  `shared`: the launch also carries the MC stage,
// which needs 128 x 64 workers; then 128 x 256 (and a launch of its own for the MC
// stage) pays only where the product is long against the stage beside it, whose
// work grows with M alone: from N = 6144 (at 8192 x 4096 the product gains 110 us
// and the separate MC launch costs about as much).
static H2Plan h2_plan(const H2Args& g, bool acc64, bool shared = false) {
  std::mutex& mu = h2_mu();
  auto& cache = h2_cache();
  const auto key = std::make_tuple(g.M, g.N, g.K, g.flags, (int)acc64 + 2 * (int)shared);
  {
    std::lock_guard<std::mutex> lk(mu);
    auto it = cache.find(key);
    if (it != cache.end()) return it->second;
  }
  const int ncu = num_cus();
  H2Plan p;
  const int small = h2_tiles(g, H2Mid::TM, H2Mid::TN), wide = h2_tiles(g, H2Wide::TM, H2Wide::TN),
            large = h2_tiles(g, H2Large::TM, H2Large::TN);
  // (the tiles 128 columns and wider read and write past an odd multiple of 64)
  const bool n128 = g.N % 128 == 0;
  if (!acc64 && n128 && 2 * large >= 3 * ncu && (!shared || g.N >= 6144))
    p = {H2Large::TN, large, 0, false};
  else if (!acc64 && n128 && !shared && 4 * wide >= 7 * ncu)
    p = {H2Wide::TN, wide, 0, false};
  else if (!acc64 && !shared && small <= ncu)
    p = {64, h2_tiles(g, H2Small::TM, H2Small::TN), 0, false};
  else
    p = h2_mid_plan(g, acc64);
  std::lock_guard<std::mutex> lk(mu);
  cache[key] = p;
  return p;
}

int gemm_h2_check(const H2Args& a) {
  const uintptr_t al16 = (uintptr_t)a.Ah | (uintptr_t)a.Al | (uintptr_t)a.Bh | (uintptr_t)a.Bl;
  if (a.M % H2_BM || a.N % 64 || a.K % H2_BK || a.M <= 0 || a.N <= 0 || a.K <= 0 ||
      a.lda % 8 || a.ldb % 8 || a.lda < a.K || a.ldb < a.K || a.ldc < a.N || !a.Ah || !a.Al ||
      !a.Bh || !a.Bl || !a.C || (a.Ch && !a.Cl) || (al16 & 15) || a.seg_chunks < 0 ||
      (a.flags & ~(BTA_GEMM_B_LOWER | BTA_GEMM_B_UPPER))) {
    set_error("gemm_h2: M%%128, N%%64, K%%32, lda/ldb%%8 must be 0, operand planes 16-byte "
              "aligned, K > 0; flags B_LOWER/B_UPPER only");
    return BTA_ERR_INVALID;
  }
  return BTA_OK;
}

int gemm_h2_candidates(const H2Args& g, bool shared, int* out, int max) {
  if (gemm_h2_check(g)) return 0;
  const int ncu = num_cus();
  const bool acc64 = g.seg_chunks > 0;
  const int slots = acc64 ? ncu : 2 * ncu;
  int k = 0;
  auto add = [&](int bn, int W, int G) {
    if (k >= max) return;
    out[3 * k] = bn;
    out[3 * k + 1] = W;
    out[3 * k + 2] = G;
    ++k;
  };
  const int total = h2_tiles(g, H2Mid::TM, H2Mid::TN);
  int last = -1;
  for (int c : {slots, 3 * slots / 4, slots / 2, 3 * slots / 8, slots / 4}) {
    const int W = std::max(1, std::min(c, total));
    if (W == last) continue;
    last = W;
    add(64, W, 1);
    const int G = h2_xcd_allowed(g, W);
    if (G > 1) add(64, W, G);
  }
  if (!acc64) {
    if (!shared) add(64, h2_tiles(g, H2Small::TM, H2Small::TN), 0);
    if (!shared && g.N % 128 == 0 && h2_tiles(g, H2Wide::TM, H2Wide::TN) >= ncu)
      add(H2Wide::TN, h2_tiles(g, H2Wide::TM, H2Wide::TN), 0);
    if (g.N % 128 == 0 && h2_tiles(g, H2Large::TM, H2Large::TN) >= ncu)
      add(H2Large::TN, h2_tiles(g, H2Large::TM, H2Large::TN), 0);
  }
  return k;
}

void gemm_h2_set_plan(const H2Args& g, bool shared, int bn, int workers, int xcd_groups) {
  const auto key =
      std::make_tuple(g.M, g.N, g.K, g.flags, (int)(g.seg_chunks > 0) + 2 * (int)shared);
  std::lock_guard<std::mutex> lk(h2_mu());
  h2_cache()[key] = H2Plan{bn, workers, xcd_groups, true};
}

int gemm_h2_shared_plan(const H2Args& a, int others, int* workers, int* xcd_groups) {
  const int rc = gemm_h2_check(a);
  if (rc) return rc;
  const H2Plan p = h2_plan(a, a.seg_chunks > 0, true);
  if (p.xcd == 0) return -1;
  *workers = p.workers;
  *xcd_groups = p.xcd;
  // One worker per CU when the other workgroups fit in one round in the CUs' second
  // slots: they then start at once instead of after the first workers (2048 x 2048
  // with 256 paired MC workgroups: 68 us with 512 workers, 50 with 256).
  const int ncu = num_cus();
  if (!p.tuned && others <= ncu && p.workers > ncu) {
    *workers = ncu;
    *xcd_groups = 1;
  }
  return BTA_OK;
}

int gemm_h2(const H2Args& args, hipStream_t s, bool shared) {
  const int rc = gemm_h2_check(args);
  if (rc) return rc;
  const bool acc64 = args.seg_chunks > 0;
  const H2Plan p = h2_plan(args, acc64, shared);
  H2Args a = args;
  a.xcd_groups = p.xcd;
  if (p.bn == H2Large::TN)
    hipLaunchKernelGGL((gemm_h2_tiles_kernel<H2Large, false>),
                       dim3(h2_tiles(a, H2Large::TM, H2Large::TN)), dim3(64 * H2Large::NW), 0, s,
                       a, num_cus());
  else if (p.bn == H2Wide::TN)
    hipLaunchKernelGGL((gemm_h2_tiles_kernel<H2Wide, false>),
                       dim3(h2_tiles(a, H2Wide::TM, H2Wide::TN)), dim3(64 * H2Wide::NW), 0, s, a,
                       num_cus());
  else if (p.xcd == 0)
    hipLaunchKernelGGL((gemm_h2_tiles_kernel<H2Small, true>),
                       dim3(h2_tiles(a, H2Small::TM, H2Small::TN)), dim3(64 * H2Small::NW), 0, s,
                       a, num_cus());
  else if (acc64)
    hipLaunchKernelGGL((gemm_h2_kernel<true>), dim3(p.workers), dim3(256), 0, s, a);
  else
    hipLaunchKernelGGL((gemm_h2_kernel<false>), dim3(p.workers), dim3(256), 0, s, a);
  BTA_LAUNCH_CHECK("gemm_h2_kernel");
  return BTA_OK;
}

// hi/lo FP16 planes of scale * X (X FP32 or FP64, rows x cols, row-major), or of
// scale * X^T when transpose is set (output cols x rows).  Zero-fills the padded
// region [rows, rows_pad) x [cols, cols_pad) of the (untransposed) index space.
template <typename T>
__global__ void split_f16_kernel(const T* __restrict__ X, int64_t ldx, int64_t rows,
                                 int64_t cols, int64_t rows_pad, int64_t cols_pad, float scale,
                                 int transpose, _Float16* __restrict__ hi,
                                 _Float16* __restrict__ lo, int64_t ldo) {
  __shared__ float tile[32][33];
  const int64_t r0 = (int64_t)blockIdx.y * 32, c0 = (int64_t)blockIdx.x * 32;
  const int tx = threadIdx.x & 31, ty = threadIdx.x >> 5;  // 256 threads: 32 x 8
  for (int i = ty; i < 32; i += 8) {
    const int64_t r = r0 + i, c = c0 + tx;
    float v = 0.0f;
    if (r < rows && c < cols) v = (float)((double)X[r * ldx + c] * (double)scale);
    tile[i][tx] = v;
  }
  __syncthreads();
  for (int i = ty; i < 32; i += 8) {
    int64_t orow, ocol;
    float x;
    if (transpose) {
      orow = c0 + i;
      ocol = r0 + tx;
      x = tile[tx][i];
      if (orow >= cols_pad || ocol >= rows_pad) continue;
    } else {
      orow = r0 + i;
      ocol = c0 + tx;
      x = tile[i][tx];
      if (orow >= rows_pad || ocol >= cols_pad) continue;
    }
    const _Float16 h = (_Float16)x;
    hi[orow * ldo + ocol] = h;
    lo[orow * ldo + ocol] = (_Float16)((x - (float)h) * 2048.0f);
  }
}

int split_f16(bool f64, const void* X, int64_t ldx, int64_t rows, int64_t cols,
              int64_t rows_pad, int64_t cols_pad, float scale, bool transpose, _Float16* hi,
              _Float16* lo, int64_t ldo, hipStream_t s) {
  if (rows < 0 || cols < 0 || rows_pad < rows || cols_pad < cols || !X || !hi || !lo ||
      ldo < (transpose ? rows_pad : cols_pad)) {
    set_error("split_f16: invalid sizes");
    return BTA_ERR_INVALID;
  }
  if (rows_pad == 0 || cols_pad == 0) return BTA_OK;
  dim3 grid((unsigned)((cols_pad + 31) / 32), (unsigned)((rows_pad + 31) / 32));
  if (f64)
    hipLaunchKernelGGL(split_f16_kernel<double>, grid, dim3(256), 0, s, (const double*)X, ldx,
                       rows, cols, rows_pad, cols_pad, scale, (int)transpose, hi, lo, ldo);
  else
    hipLaunchKernelGGL(split_f16_kernel<float>, grid, dim3(256), 0, s, (const float*)X, ldx,
                       rows, cols, rows_pad, cols_pad, scale, (int)transpose, hi, lo, ldo);
  BTA_LAUNCH_CHECK("split_f16_kernel");
  return BTA_OK;
}

}  // namespace bta

extern "C" int bta_split_f16(int32_t src_f64, const void* X, int64_t ldx, int64_t rows,
                             int64_t cols, int64_t rows_pad, int64_t cols_pad, float scale,
                             int32_t transpose, void* hi, void* lo, int64_t ldo,
                             bta_stream_t stream) {
  return bta::split_f16(src_f64 != 0, X, ldx, rows, cols, rows_pad, cols_pad, scale,
                        transpose != 0, (_Float16*)hi, (_Float16*)lo, ldo,
                        (hipStream_t)stream);
}

extern "C" int bta_gemm_f16x3(int32_t flags, int64_t M, int64_t N, int64_t K, double alpha,
                              const void* a_hi, const void* a_lo, int64_t lda,
                              const float* a_row_scale, float a_scale, const void* b_hi,
                              const void* b_lo, int64_t ldb, float b_scale, float* C,
                              int64_t ldc, void* c_hi, void* c_lo, float c_scale,
                              int32_t k_segment, bta_stream_t stream) {
  if (M > (1 << 30) || N > (1 << 30) || K > (1 << 30) || k_segment < 0 || k_segment % 32) {
    bta::set_error("bta_gemm_f16x3: sizes beyond 2^30 or k_segment not a multiple of 32");
    return BTA_ERR_INVALID;
  }
  bta::H2Args a{};
  a.Ah = (const _Float16*)a_hi;
  a.Al = (const _Float16*)a_lo;
  a.Bh = (const _Float16*)b_hi;
  a.Bl = (const _Float16*)b_lo;
  a.C = C;
  a.Ch = (_Float16*)c_hi;
  a.Cl = (_Float16*)c_lo;
  a.a_row_scale = a_row_scale;
  a.a_scale = a_scale;
  a.b_scale = b_scale;
  a.c_scale = c_scale;
  a.lda = lda;
  a.ldb = ldb;
  a.ldc = ldc;
  a.M = (int)M;
  a.N = (int)N;
  a.K = (int)K;
  a.flags = flags;
  a.alpha = alpha;
  a.seg_chunks = k_segment / 32;
  return bta::gemm_h2(a, (hipStream_t)stream);
}
