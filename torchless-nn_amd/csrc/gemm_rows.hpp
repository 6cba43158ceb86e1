// Host interface of gemm_rows.hip.
#pragma once

#include "gemm_common.hpp"

namespace tl {

// A choice of gemm_rows_kernel: its tile (an index into the tile table; < 0: leave the product
// to the other kernels), over how many workgroups a tile's K is split, and its modelled time.
struct RowsPlan {
  int tile = -1, splits = 1;
  float us = 0;
};
// The choice for an unbatched product [M, K] x [N, K] whose K is a multiple of 128 bytes (rules
// from measurements): bf16 operands, and fp32 ones (whose time competes with SplitPlan's).
// `can_stream`: whether gemm_skinny_stream_kernel can have its workspace.
RowsPlan gemm_rows_plan(int64_t M, int64_t N, int64_t K, int cus, bool can_stream);
RowsPlan gemm_rows_plan_f32(int64_t M, int64_t N, int64_t K, int cus);
// Runs it. Operands as gemm_mfma_kernel / gemm_mfma_f32_kernel take them, batch 1.
int gemm_rows_launch(tl_ctx* ctx, GemmParams p, RowsPlan plan, bool f32in, bool f32out, int family,
                     double flops, double bytes);

}  // namespace tl
