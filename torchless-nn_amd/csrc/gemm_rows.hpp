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
// The choice for an unbatched bf16 product [M, K] x [N, K], K % 64 == 0 (a rule from measurements).
RowsPlan gemm_rows_plan(int64_t M, int64_t N, int64_t K, int cus);
// Runs it. Operands as gemm_mfma_kernel takes them, batch 1.
int gemm_rows_launch(tl_ctx* ctx, GemmParams p, RowsPlan plan, bool f32out, int family,
                     double flops, double bytes);

}  // namespace tl
