// One 32 x 32 tile of an FP64 product per workgroup, for gemm_w.hip and the kernels
// that fuse it with their own work.
//
// The KS waves of a workgroup share the tile and split its K range in chunks of 16
// dealt round-robin, each wave with all of the tile's accumulators; the partial
// tiles are added through LDS in a fixed order at the end.  That cuts the longest
// serial K range KS-fold (a triangular product's longest tile has twice the average
// length and sits on one CU) and gives 8 times as many workgroups.  Every wave
// stages its own chunks by direct-to-LDS loads through a ring of two stages, so
// there is no barrier in the loop, only the wave's own vmcnt wait.
//
// What bounds it: the operands are re-read per tile, 32 bytes a cycle and CU
// against the 64 cycles of a 16x16x4 product, so large products stay 1.55 x off
// the matrix rate and with gemm_d (1.16 x).  Fragments loaded straight to
// registers were slower (16 rows x 64 bytes per load instruction, ~56 cycles each
// in the address path, against 8 rows x 128 bytes here): 125 against 101 us at
// 1024 x 2048; chunks of 32, a third stage, and 32 x 64 or 64 x 64 tiles leave one
// wave per SIMD and were slower too (117, 125, 110, 123 us).
//
// K assignment: piece c of a chunk (k = 2 c, 2 c + 1) goes to lane group c % 4 for
// both operands.  With B K x N a lane reads two neighbouring columns, so column
// block ni holds the columns 2 l16 + ni of the tile.
#pragma once
#include "bta_common.h"
#include "gemm.h"
#include "gemm_d.h"
#include "gemm_tile.h"

namespace bta {

template <int FM, int FN, int CK, int ST>
struct WCfg {  // FM x FN fragments, chunks of CK, ST stages
  static constexpr int TM = 16 * FM, TN = 16 * FN;
  static constexpr int RA = TM * CK * 8, RB = TN * CK * 8;  // bytes per stage
  static constexpr int STAGE = RA + RB;
  static constexpr int LA = RA / 1024, LB = RB / 1024;  // 1 KiB wave loads
  static constexpr int CPR = CK / 2;                    // 16-byte slots of a K-contiguous row
  static_assert(FM * FN * 16 * 16 * 8 <= ST * STAGE, "the reduction reuses the ring");
};

// Slot of 16-byte piece c of a K-contiguous stage row r: c ^ (r mod slots), so
// that eight rows' pieces c fall in distinct slots of a 128-byte line.
template <int CPR>
__device__ __forceinline__ int w_slot(int c, int r) { return c ^ (r & (CPR - 1)); }

// The products A[row0 .., kb:ke] op(B)[kb:ke, col0 ..] of one tile by the KS waves of a
// workgroup, their partial tiles left in lds as doubles [wave][fragment][q][lane]
// (w_sum adds them; fragment f = (f / FN, f % FN), accumulator layout); ends with a
// barrier.  lds: w_lds bytes.  ke - kb a multiple of CK.
template <int FM, int FN, int KS, int CK, int ST, bool BKN>
__device__ __forceinline__ void w_partials(const double* A, int64_t lda, const double* B,
                                           int64_t ldb, int row0, int col0, int kb, int ke,
                                           unsigned char* lds) {
  static_assert(!BKN || FN % 2 == 0, "column pairs");
  using C = WCfg<FM, FN, CK, ST>;
  const int lane = threadIdx.x & 63, wv = wave_uniform(threadIdx.x >> 6);
  const int l16 = lane & 15, gq = lane >> 4;
  const int nk = ((ke - kb) / CK - wv + KS - 1) / KS;  // this wave's chunks wv, wv + KS, ...
  unsigned char* ring = lds + wv * ST * C::STAGE;

  // wave load j: 1 KiB of consecutive stage rows, (lane -> row, slot)
  const double* src[C::LA + C::LB];
  int64_t step[2] = {(int64_t)KS * CK, BKN ? (int64_t)KS * CK * ldb : (int64_t)KS * CK};
  {
    constexpr int RPL = 64 / C::CPR;  // rows per load of a K-contiguous operand
    const int r = lane / C::CPR, sl = lane % C::CPR;
#pragma unroll
    for (int j = 0; j < C::LA; ++j) {
      const int rr = j * RPL + r;
      src[j] = A + (int64_t)(row0 + rr) * lda + kb + wv * CK + 2 * w_slot<C::CPR>(sl, rr);
    }
#pragma unroll
    for (int j = 0; j < C::LB; ++j) {
      if (BKN) {  // stage rows are k, TN doubles each
        const int e = j * 128 + lane * 2;
        src[C::LA + j] = B + (int64_t)(kb + wv * CK + e / C::TN) * ldb + col0 + e % C::TN;
      } else {
        const int rr = j * RPL + r;
        src[C::LA + j] =
            B + (int64_t)(col0 + rr) * ldb + kb + wv * CK + 2 * w_slot<C::CPR>(sl, rr);
      }
    }
  }
  auto issue = [&](int ci) {
    unsigned char* st = ring + (ci % ST) * C::STAGE;
#pragma unroll
    for (int j = 0; j < C::LA + C::LB; ++j) {
      const double* p = src[j] + ci * step[j >= C::LA];
      __builtin_amdgcn_global_load_lds(p, (lds_ptr_t)(st + j * 1024), 16, 0, 0);
    }
  };
  // fragments of a stage: a[mi][u], b[ni][u] = the pieces c = 4 u + g (k = 2 c,
  // 2 c + 1) of the lane's rows; K-major B: b[2 f + e'][..] see mul
  v2d a[FM][CK / 8], b[FN][CK / 8];
  auto read = [&](int ci) {
    const unsigned char* st = ring + (ci % ST) * C::STAGE;
#pragma unroll
    for (int mi = 0; mi < FM; ++mi)
#pragma unroll
      for (int u = 0; u < CK / 8; ++u)
        a[mi][u] = lds_read_b128<0>(lds_addr(
            st + (16 * mi + l16) * CK * 8 + w_slot<C::CPR>(4 * u + gq, 16 * mi + l16) * 16));
    const unsigned char* sb = st + C::RA;
#pragma unroll
    for (int ni = 0; ni < FN; ++ni)
#pragma unroll
      for (int u = 0; u < CK / 8; ++u) {
        if (BKN)  // row k = 8 u + 2 g + (ni & 1), columns 32 (ni / 2) + 2 l16, + 1
          b[ni][u] = lds_read_b128<0>(lds_addr(
              sb + ((8 * u + 2 * gq + (ni & 1)) * C::TN + 32 * (ni / 2) + 2 * l16) * 8));
        else
          b[ni][u] = lds_read_b128<0>(lds_addr(
              sb + (16 * ni + l16) * CK * 8 + w_slot<C::CPR>(4 * u + gq, 16 * ni + l16) * 16));
      }
    lds_frag_wait();
#pragma unroll
    for (int mi = 0; mi < FM; ++mi)
#pragma unroll
      for (int u = 0; u < CK / 8; ++u) __asm__ __volatile__("" : "+v"(a[mi][u]));
#pragma unroll
    for (int ni = 0; ni < FN; ++ni)
#pragma unroll
      for (int u = 0; u < CK / 8; ++u) __asm__ __volatile__("" : "+v"(b[ni][u]));
  };
  v4d acc[FM][FN];
#pragma unroll
  for (int mi = 0; mi < FM; ++mi)
#pragma unroll
    for (int ni = 0; ni < FN; ++ni) acc[mi][ni] = (v4d)(0.0);
  auto mul = [&]() {
#pragma unroll
    for (int u = 0; u < CK / 8; ++u)
#pragma unroll
      for (int e = 0; e < 2; ++e)
#pragma unroll
        for (int mi = 0; mi < FM; ++mi)
#pragma unroll
          for (int ni = 0; ni < FN; ++ni) {
            const double bv = BKN ? b[(ni & ~1) + e][u][ni & 1] : b[ni][u][e];
            acc[mi][ni] =
                __builtin_amdgcn_mfma_f64_16x16x4f64(a[mi][u][e], bv, acc[mi][ni], 0, 0, 0);
          }
  };
#pragma unroll
  for (int ci = 0; ci < ST; ++ci)
    if (ci < nk) issue(ci);
  constexpr int LPC = C::LA + C::LB;
  for (int it = 0; it < nk; ++it) {
    // chunk it has landed when only the later chunks' loads are outstanding
    const int later = min(ST - 1, nk - 1 - it);
    if (ST > 2 && later >= 2) d_wait_vmcnt<(ST > 2 ? 2 : 0) * LPC>();
    else if (later >= 1) d_wait_vmcnt<LPC>();
    else d_wait_vmcnt<0>();
    __builtin_amdgcn_sched_barrier(0);
    __asm__ __volatile__("" ::: "memory");
    read(it);
    __builtin_amdgcn_sched_barrier(0);
    if (it + ST < nk) issue(it + ST);
    __builtin_amdgcn_sched_barrier(0);
    mul();
  }
  // the partial tiles over the ring
  double* red = (double*)lds;
  __syncthreads();
#pragma unroll
  for (int f = 0; f < FM * FN; ++f)
#pragma unroll
    for (int q = 0; q < 4; ++q)
      red[((wv * FM * FN + f) * 4 + q) * 64 + lane] = acc[f / FN][f % FN][q];
  __syncthreads();
}

// Entry (f, q, lane) of the tile: the waves' partials in wave order.
template <int FM, int FN, int KS>
__device__ __forceinline__ double w_sum(const double* red, int f, int q, int lane) {
  double v = red[(f * 4 + q) * 64 + lane];
#pragma unroll
  for (int w = 1; w < KS; ++w) v += red[((w * FM * FN + f) * 4 + q) * 64 + lane];
  return v;
}

template <int FM, int FN, int KS, int CK, int ST>
constexpr int w_lds() {
  return KS * ST * WCfg<FM, FN, CK, ST>::STAGE;
}

// Tile t0 of product `batch`; ncu: workgroups of one round.
template <int FM, int FN, int KS, int CK, int ST, bool BKN>
__device__ __forceinline__ void gemm_w_body(const GemmArgs& g, int t0, int64_t batch, int ncu,
                                            unsigned char* lds) {
  using C = WCfg<FM, FN, CK, ST>;
  const double* A = (const double*)g.A + batch * g.sA;
  const double* B = (const double*)g.B + batch * g.sB;
  const int MT = g.M / C::TM, NT = g.N / C::TN;
  // tiles longest first; odd rounds of one workgroup per CU run backwards, so a
  // CU's first two workgroups hold a long and a short tile
  const int total = MT * NT;
  const int rd = t0 / ncu;
  if (rd & 1) t0 = rd * ncu + min(ncu, total - rd * ncu) - 1 - (t0 - rd * ncu);
  int tm, tn;
  decode_tile(t0, g.flags, MT, NT, tm, tn);
  int kb = 0, ke = g.K;
  if (g.flags & BTA_GEMM_B_LOWER) ke = min(ke, (tn + 1) * C::TN);
  if (g.flags & BTA_GEMM_B_UPPER) kb = max(kb, tn * C::TN);
  const int lane = threadIdx.x & 63, wv = wave_uniform(threadIdx.x >> 6);
  const int l16 = lane & 15, gq = lane >> 4;
  const int row0 = tm * C::TM, col0 = tn * C::TN;
  w_partials<FM, FN, KS, CK, ST, BKN>(A, g.lda, B, g.ldb, row0, col0, kb, ke, lds);
  const double* red = (const double*)lds;
  double* Cp = (double*)g.C + batch * g.sC;
  const double* C0 = g.C0 ? (const double*)g.C0 + batch * g.sC0 : nullptr;
  // slice wv finishes the fragments wv, wv + KS, ...
#pragma unroll
  for (int f0 = 0; f0 < FM * FN; f0 += KS) {
    const int f = f0 + wv;
    if (FM * FN % KS && f >= FM * FN) break;
    const int mi = f / FN, ni = f % FN;
    const int64_t col = col0 + (BKN ? 32 * (ni / 2) + 2 * l16 + (ni & 1) : 16 * ni + l16);
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      double v = w_sum<FM, FN, KS>(red, f, q, lane);
      const int64_t row = row0 + 16 * mi + Mfma<double>::row(gq, q);
      v *= g.alpha;
      if (C0) v += g.beta * C0[row * g.ldc0 + col];
      Cp[row * g.ldc + col] = v;
    }
  }
}

}  // namespace bta
