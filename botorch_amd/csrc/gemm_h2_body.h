// Split-FP16 GEMM worker body shared by gemm_h2_kernel and the fused
// adjoint-GEMM + MC launch of the qLogNEI step (the algorithm is described at
// the top of gemm_h2.hip).
#pragma once
#include "bta_common.h"
#include "gemm.h"
#include "gemm_d.h"
#include "gemm_tile.h"
#include "kernels.h"

namespace bta {

typedef _Float16 half8 __attribute__((ext_vector_type(8)));

constexpr int H2_BM = 128;       // row tile of the worker schedules (H2Mid)
constexpr int H2_BK = 32;        // K per chunk (one MFMA K-step)
constexpr int H2_ROWB = 128;     // bytes per stage row: 32 halfs of each plane
constexpr double H2_LO = 1.0 / 2048.0;  // weight of the lo planes (stored as 2^11 (x - hi))

// s_waitcnt on the vector-memory counter only (expcnt, lgkmcnt left open)
template <int N>
__device__ __forceinline__ void wait_vmcnt() {
  static_assert(N >= 0 && N < 64, "vmcnt range");
  __builtin_amdgcn_s_waitcnt((N & 15) | (7 << 4) | (15 << 8) | ((N >> 4) << 14));
}

template <int OFF>
__device__ __forceinline__ half8 h2_read(uint32_t a) {
  half8 v;
  __asm__ __volatile__("ds_read_b128 %0, %1 offset:%2" : "=v"(v) : "v"(a), "i"(OFF));
  return v;
}
__device__ __forceinline__ void h2_tie(half8& v) { __asm__ __volatile__("" : "+v"(v)); }

// WM x WN waves of FM x FN 16 x 16 fragments, S ring stages.  A stage row is one
// row's chunk of both planes, [hi | lo], 128 bytes.
template <int WM, int WN, int FM, int FN, int S>
struct H2Cfg {
  static constexpr int TM = WM * FM * 16, TN = WN * FN * 16, NW = WM * WN;
  static constexpr int RA = TM * 128, STAGE = (TM + TN) * 128, STAGES = S;
  static constexpr int LW = (TM + TN) / 8 / NW;  // 1 KiB loads per wave and chunk
  static_assert((TM + TN) / 8 % NW == 0, "wave loads must split over the waves");
  static_assert(128 % TM == 0, "M is a multiple of 128");
};

// The tiles (TM x TN): see the comment at the top of gemm_h2.hip.
typedef H2Cfg<2, 2, 2, 2, 3> H2Small;   // 64 x 64
typedef H2Cfg<2, 2, 4, 2, 3> H2Mid;     // 128 x 64
typedef H2Cfg<4, 4, 2, 2, 3> H2Wide;    // 128 x 128
typedef H2Cfg<2, 4, 4, 4, 3> H2Large;   // 128 x 256

// F fragments, 2 KiB (16 rows) apart
template <int F>
__device__ __forceinline__ void h2_frag(uint32_t a, half8 (&x)[F]) {
  static_assert(F <= 4, "fragments per wave edge");
  if constexpr (F > 0) x[0] = h2_read<0>(a);
  if constexpr (F > 1) x[1] = h2_read<2048>(a);
  if constexpr (F > 2) x[2] = h2_read<4096>(a);
  if constexpr (F > 3) x[3] = h2_read<6144>(a);
}

// The main loop and epilogue of one output tile (tm, tn) with the ring in lds
// (S * STAGE bytes, 1 KiB aligned).  Every tile shape sums an element's products
// in the same order: per chunk of 32 ascending k, lo x hi then hi x lo into one
// FP32 sum, hi x hi into the other.  ACC64: both are added into FP64 sums and
// restarted every g.seg_chunks chunks.
template <bool ACC64 = false, int WM, int WN, int FM, int FN, int S>
__device__ __forceinline__ void gemm_h2_tile(H2Cfg<WM, WN, FM, FN, S>, const H2Args& g,
                                             const int tm, const int tn, unsigned char* lds) {
  using C = H2Cfg<WM, WN, FM, FN, S>;
  const int lane = threadIdx.x & 63, wv = wave_uniform(threadIdx.x >> 6);
  const int wy = wv / WN, wx = wv % WN, l16 = lane & 15, gq = lane >> 4;
  int kb = 0, ke = g.K;
  if (g.flags & BTA_GEMM_B_LOWER) ke = min(ke, (tn + 1) * C::TN);
  if (g.flags & BTA_GEMM_B_UPPER) kb = max(kb, tn * C::TN);
  kb = kb / H2_BK * H2_BK;
  ke = (ke + H2_BK - 1) / H2_BK * H2_BK;
  const int row0 = tm * C::TM, col0 = tn * C::TN;
  const int nk = ke > kb ? (ke - kb) / H2_BK : 0;

  // direct loads: eight rows a wave load; lane -> (row lane / 8, slot lane % 8),
  // whose piece c is 0..3 of the hi plane or 4..7 of the lo plane.  Columns past N
  // (the last tile of a wide shape) read the ones 128 earlier.
  const int c = (lane & 7) ^ (lane >> 3);
  const _Float16* src[C::LW];
#pragma unroll
  for (int j = 0; j < C::LW; ++j) {
    const int gi = wv * C::LW + j, r = gi * 8 + (lane >> 3), ko = kb + (c & 3) * 8;
    if (gi < C::TM / 8) {
      src[j] = (c & 4 ? g.Al : g.Ah) + (int64_t)(row0 + r) * g.lda + ko;
    } else {
      int n = col0 + r - C::TM;
      if (C::TN > 128 && n >= g.N) n -= 128;
      src[j] = (c & 4 ? g.Bl : g.Bh) + (int64_t)n * g.ldb + ko;
    }
  }
  auto issue = [&](int ci) {
    unsigned char* st = lds + (ci % S) * C::STAGE + wv * C::LW * 1024;
#pragma unroll
    for (int j = 0; j < C::LW; ++j) {
      // (a named pointer: the builtin rejects the expression in the host pass)
      const _Float16* p = src[j] + ci * H2_BK;
      __builtin_amdgcn_global_load_lds(p, (lds_ptr_t)(st + j * 1024), 16, 0, 0);
    }
  };
  v4f acc[FM][FN], accx[FM][FN];
#pragma unroll
  for (int mi = 0; mi < FM; ++mi)
#pragma unroll
    for (int ni = 0; ni < FN; ++ni) acc[mi][ni] = accx[mi][ni] = (v4f)(0.0f);
  double acc64[ACC64 ? FM : 1][ACC64 ? FN : 1][4] = {};
  const int seg = ACC64 ? g.seg_chunks : 1;  // chunks per FP64 add
  // fragment reads: row l16 of a 16-row block, piece gq in its slot; the lo
  // plane's piece gq + 4 lies at the address with bit 6 flipped
  const int foff = l16 * H2_ROWB + ((gq ^ (l16 & 7)) << 4);

#pragma unroll
  for (int ci = 0; ci < S - 1; ++ci)
    if (ci < nk) issue(ci);
  for (int it = 0; it < nk; ++it) {
    // this wave's loads of chunk it have landed once at most
    // min(S - 2, nk - 1 - it) later chunks remain outstanding
    static_assert(S == 3, "the vmcnt levels assume 3 stages");
    if (it + 1 < nk) wait_vmcnt<C::LW>();
    else wait_vmcnt<0>();
    // every wave's loads of chunk it landed and every wave is done with chunk
    // it - 1.  A bare s_barrier: the fence of __syncthreads would also wait for
    // the loads still in flight; the empty asm statements keep the compiler
    // from moving LDS accesses across it.
    // sched_barrier(0): the compiler moves nothing across, in particular no
    // LDS read of this chunk above the wait and the barrier (another wave's
    // direct loads fill part of the stage, and only the barrier orders them)
    __builtin_amdgcn_sched_barrier(0);
    __asm__ __volatile__("" ::: "memory");
    __builtin_amdgcn_s_barrier();
    __asm__ __volatile__("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
    if (it + S - 1 < nk) issue(it + S - 1);
    const unsigned char* cur = lds + (it % S) * C::STAGE;
    // fragment reads as inline asm (see lds_read_b128): no compiler-added
    // vmcnt(0) for the direct loads in flight
    half8 ah[FM], al[FM], bh[FN], bl[FN];
    const uint32_t aa = lds_addr(cur + wy * FM * 2048 + foff);
    const uint32_t ba = lds_addr(cur + C::RA + wx * FN * 2048 + foff);
    h2_frag(aa ^ 64, al);
    h2_frag(ba, bh);
    h2_frag(aa, ah);
    h2_frag(ba ^ 64, bl);
    // LDS reads return in order: the first FM + FN are in once FM + FN remain
    __asm__ __volatile__("s_waitcnt lgkmcnt(%0)" ::"i"(FM + FN) : "memory");
#pragma unroll
    for (int f = 0; f < FM; ++f) h2_tie(al[f]);
#pragma unroll
    for (int f = 0; f < FN; ++f) h2_tie(bh[f]);
    // accx += A_lo B_hi + A_hi B_lo, acc += A_hi B_hi; three passes over the
    // fragments, so no MFMA waits on the one before it, the first of them while
    // the other two operands are still on their way
#pragma unroll
    for (int mi = 0; mi < FM; ++mi)
#pragma unroll
      for (int ni = 0; ni < FN; ++ni)
        accx[mi][ni] =
            __builtin_amdgcn_mfma_f32_16x16x32_f16(al[mi], bh[ni], accx[mi][ni], 0, 0, 0);
    __builtin_amdgcn_sched_barrier(0);
    lds_frag_wait();
#pragma unroll
    for (int f = 0; f < FM; ++f) h2_tie(ah[f]);
#pragma unroll
    for (int f = 0; f < FN; ++f) h2_tie(bl[f]);
#pragma unroll
    for (int mi = 0; mi < FM; ++mi)
#pragma unroll
      for (int ni = 0; ni < FN; ++ni)
        acc[mi][ni] = __builtin_amdgcn_mfma_f32_16x16x32_f16(ah[mi], bh[ni], acc[mi][ni], 0, 0, 0);
#pragma unroll
    for (int mi = 0; mi < FM; ++mi)
#pragma unroll
      for (int ni = 0; ni < FN; ++ni)
        accx[mi][ni] =
            __builtin_amdgcn_mfma_f32_16x16x32_f16(ah[mi], bl[ni], accx[mi][ni], 0, 0, 0);
    if constexpr (ACC64) {
      if ((it + 1) % seg == 0 || it + 1 == nk) {
#pragma unroll
        for (int mi = 0; mi < FM; ++mi)
#pragma unroll
          for (int ni = 0; ni < FN; ++ni) {
#pragma unroll
            for (int q = 0; q < 4; ++q)
              acc64[mi][ni][q] += (double)acc[mi][ni][q] + H2_LO * (double)accx[mi][ni][q];
            acc[mi][ni] = accx[mi][ni] = (v4f)(0.0f);
          }
      }
    }
  }
  // all waves done reading the ring before the next tile's loads overwrite it
  __syncthreads();
  const double bs = (double)g.b_scale;
#pragma unroll
  for (int mi = 0; mi < FM; ++mi)
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int64_t row = row0 + (wy * FM + mi) * 16 + Mfma<float>::row(gq, q);
      const double f =
          g.alpha / ((double)g.a_scale * (g.a_row_scale ? (double)g.a_row_scale[row] : 1.0) * bs);
#pragma unroll
      for (int ni = 0; ni < FN; ++ni) {
        const int64_t col = col0 + (wx * FN + ni) * 16 + l16;
        if (C::TN > 128 && col >= g.N) continue;
        const double sum = ACC64 ? acc64[ACC64 ? mi : 0][ACC64 ? ni : 0][q]
                                 : (double)acc[mi][ni][q] + H2_LO * (double)accx[mi][ni][q];
        const float v = (float)(sum * f);
        g.C[row * g.ldc + col] = v;
        if (g.Ch) {
          const float x = v * g.c_scale;
          const _Float16 h = (_Float16)x;
          g.Ch[row * g.ldc + col] = h;
          g.Cl[row * g.ldc + col] = (_Float16)((x - (float)h) * 2048.0f);
        }
      }
    }
}

// Worker w of W: the tiles h2_tile_of(jj, w, W), jj = 0, 1, ... of the
// problem's longest-first tile order.  With g.xcd_groups = G > 1 (triangular
// B, tiles ordered column strip by column strip, NT a multiple of 2 G), the
// workers form G groups by w % G - the XCD a workgroup is dispatched to - and
// group x takes the strips x, 2G - 1 - x, 2G + x, 4G - 1 - x, ... of that order
// (a snake, so that every group's strips add up to the same K length), so all
// row tiles of a strip of B run on one XCD and read the strip through one L2;
// within the group the tiles are dealt as above over its W / G workers (W a
// multiple of G), still longest first.
template <bool ACC64 = false>
__device__ __forceinline__ void gemm_h2_body(const H2Args& g, int w, int W, unsigned char* lds) {
  const int MT = g.M / H2Mid::TM, NT = g.N / H2Mid::TN;
  const int G = g.xcd_groups;
  if (G > 1) {
    const int x = w % G, lw = w / G, Wx = W / G;
    const int total = (NT / G) * MT;  // MT row tiles of each of the group's NT / G strips
    for (int jj = 0;; ++jj) {
      const int u = h2_tile_of(jj, lw, Wx);
      if (jj * Wx >= total) break;
      if (u >= total) continue;
      const int j = u / MT;
      const int strip = j * G + ((j & 1) ? G - 1 - x : x);
      const int t = strip * MT + u % MT;
      int tm, tn;
      decode_tile(t, g.flags, MT, NT, tm, tn);
      gemm_h2_tile<ACC64>(H2Mid(), g, tm, tn, lds);
    }
    return;
  }
  const int total = MT * NT;
  for (int jj = 0;; ++jj) {
    const int t = h2_tile_of(jj, w, W);
    if (jj * W >= total) break;
    if (t >= total) continue;
    int tm, tn;
    decode_tile(t, g.flags, MT, NT, tm, tn);
    gemm_h2_tile<ACC64>(H2Mid(), g, tm, tn, lds);
  }
}

// Worker w of W over a list of tiles of many problems: tiles[t] = (problem,
// tm, tn, -), listed longest K range first; problem p's arguments are tab[p].
__device__ __forceinline__ void gemm_h2_list_body(const H2Args* __restrict__ tab,
                                                  const int4* __restrict__ tiles, int total,
                                                  int w, int W, unsigned char* lds) {
  for (int jj = 0;; ++jj) {
    const int t = h2_tile_of(jj, w, W);
    if (jj * W >= total) break;
    if (t >= total) continue;
    const int4 e = tiles[t];
    const H2Args g = tab[e.x];
    gemm_h2_tile(H2Mid(), g, e.y, e.z, lds);
  }
}

}  // namespace bta
