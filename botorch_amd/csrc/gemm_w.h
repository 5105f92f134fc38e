// Interface of the small-tile FP64 GEMM (gemm_w.hip).
#pragma once
#include "gemm.h"

namespace bta {

// M, N, K multiples of 32, 16-byte aligned operands with even strides, no flags
// but B_LOWER, B_UPPER and B_KN.
bool gemm_w_supported(const GemmArgs& g);
// Whether the small tiles are the faster ones for this output size.
bool gemm_w_preferred(int64_t M, int64_t N, int batch);
int gemm_w(const GemmArgs& g, int batch, hipStream_t s);

}  // namespace bta
