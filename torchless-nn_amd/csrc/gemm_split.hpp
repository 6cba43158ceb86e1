// Host interface of gemm_split.hip.
#pragma once

#include "gemm_common.hpp"

namespace tl {

// A choice of gemm_split_kernel: its tile (an index into the tile table; < 0: leave the product
// to the other kernels), how many tiles of the order take one workgroup each (each of the others
// takes `splits`, with a part of K each), and the modelled time.
struct SplitPlan {
  int tile = -1, full = 0, splits = 1;
  float us = 0;
};
// The choice for an unbatched fp32 product [M, K] x [N, K], K % 32 == 0.
SplitPlan gemm_split_plan(int64_t M, int64_t N, int64_t K, int cus);
// Runs it. Operands as gemm_mfma_f32_kernel takes them, batch 1.
int gemm_split_launch(tl_ctx* ctx, GemmParams p, SplitPlan plan, bool f32out, int family,
                      double flops, double bytes);

}  // namespace tl
