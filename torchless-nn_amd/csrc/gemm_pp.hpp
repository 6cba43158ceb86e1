// Host interface of gemm_pp.hip.
#pragma once

#include "gemm_common.hpp"

namespace tl {

// Whether gemm_pp_kernel takes an unbatched bf16 product with bf16 output, K % 64 == 0 and the
// given EpiKind (a measured rule).
bool gemm_pp_takes(int64_t M, int64_t N, int64_t K, int epi, int cus);
int gemm_pp_launch(tl_ctx* ctx, GemmParams p, int family, double flops, double bytes);

}  // namespace tl
