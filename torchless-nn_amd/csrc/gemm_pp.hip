// gemm_pp_kernel: large bf16 products on 256x256 tiles whose two halves take turns at the matrix
// cores. gemm_dma_kernel's eight waves all read their fragments from LDS at the start of a K step
// and all run MFMAs after, so the matrix cores idle through the reads (65% busy at 8192^3). Here
// the four waves of the upper 128 rows (one per SIMD) and the four of the lower run half a phase
// apart: while one half reads 12 fragments per wave, the other runs 32 MFMAs, then they meet at a
// barrier and swap.
//
// K steps of 64, two LDS stages of 64 KB, two phases (32-wide K halves h) per step. With intervals
// between barriers numbered 4 t + i in step t, the upper half reads h = 0 in 4t, computes in 4t + 1,
// reads h = 1 in 4t + 2, computes in 4t + 3; the lower half does the same one interval later. The
// stage of step t + 1 held step t - 1, read last by the lower half in 4t - 1, so loads for step
// t + 1 may be issued from 4t on and have to be done when 4t + 4 begins: the upper waves issue
// theirs (tile A) in 4t and wait for them at the end of 4t + 3, the lower waves theirs (tile B) in
// 4t + 1 and wait in 4t + 3.
//
// us against the tiles used before: 8192^3 801 -> 757 (1453 TFLOP/s), 8192 x 32768 x 2048 (gated)
// 846 -> 794, 8192 x 2048 x 2048 78 -> 64, 8192 x 4096 x 1024 80 -> 64, 8192 x 6144 x 768 (GeLU)
// 110 -> 92, 8192 x 50257 x 768 685 -> 668 (the LM head in the GPT-2 forward, kernel traces in turn),
// 8192 x 2048 x 16384 441 -> 433. What bounds it is the LDS: with the loads left out it runs at 2.1 PFLOP/s, with all loads from the same cached lines
// at 1.53, so the 64 KB a step writes into LDS beside the 192 KB it reads costs more than their
// latency. Tried: loads among the MFMAs instead of the reads (1429 TFLOP/s at 8192^3, 460 us at K =
// 16384), five 32-wide stages (twice the lookahead, 1314), no s_setprio (1354), a 256x192 tile (ties
// with the 128-row tiles where 256x256 does not fill its rounds).
#include <algorithm>
#include <type_traits>

#include "gemm_epilogue.hpp"
#include "gemm_pp.hpp"

namespace tl {

__device__ __forceinline__ void pp_barrier() {
  __builtin_amdgcn_sched_barrier(0);
  asm volatile("s_barrier" ::: "memory");
  __builtin_amdgcn_sched_barrier(0);
}

// EARLY: a step's loads are issued before its first fragment reads instead of after them.
template <bool EARLY>
__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(2, 2)))
void gemm_pp_kernel(GemmParams p) {
  constexpr int BM = 256, BN = 256, BK = 64, WM = 128, WN = 64, TM = 8, TN = 4;
  constexpr int SZ = (BM + BN) * BK;
  __shared__ __attribute__((aligned(16))) bf16_t S0[SZ];
  __shared__ __attribute__((aligned(16))) bf16_t S1[SZ];

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave >> 2, wn = wave & 3;
  const bool upper = wm == 0;
  int tm, tn;
  map_tile(blockIdx.x, p, tm, tn);
  const int64_t m0 = (int64_t)tm * BM, n0 = (int64_t)tn * BN;
  // the upper waves load the A tile, the lower ones the B tile: 8 groups of 8 rows x 8 chunks
  // each, lane l filling row l / 8, slot l % 8 with chunk (l % 8) ^ (row % 8); rows past M or N
  // are clamped to the last one (computed, never stored)
  const bf16_t* src = upper ? (const bf16_t*)p.A + m0 * p.lda : (const bf16_t*)p.B + n0 * p.ldb;
  const int g0 = 8 * wn;  // this wave's first group of its tile
  uint32_t off[8];
  {
    const int last = (int)min((int64_t)256, upper ? p.M - m0 : p.N - n0) - 1;
    const int64_t ld = upper ? p.lda : p.ldb;
    const int rin = lane >> 3, c = (lane & 7) ^ rin;
#pragma unroll
    for (int j = 0; j < 8; ++j) off[j] = (uint32_t)(min(8 * (g0 + j) + rin, last) * ld + c * 8);
  }
  const int nk = (int)(p.K / BK);
  // this half's loads of step t (of the last one again past the end, into a free stage)
  auto load = [&](auto up_tag, bf16_t* S, int t) {
    constexpr bool UP = decltype(up_tag)::value;
    const bf16_t* from = src + (int64_t)min(t, nk - 1) * BK;
    const uint32_t to = lds_offset(S) + ((UP ? 0 : 32) + g0) * 1024;
#pragma unroll
    for (int j = 0; j < 8; ++j) dma_load16(from + off[j], to + j * 1024);
  };

  f32x4 acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  const int fr = lane & 15, fc = lane >> 4;
  const int a_frag = (wm * WM + fr) * BK, b_frag = BM * BK + (wn * WN + fr) * BK;
  bf16x8 af[TM], bfr[TN];
  auto read = [&](const bf16_t* S, int h) {
    const int sw = ((h * 4 + fc) ^ (fr & 7)) << 3;
#pragma unroll
    for (int j = 0; j < TN; ++j) bfr[j] = *reinterpret_cast<const bf16x8*>(&S[b_frag + j * 16 * BK + sw]);
#pragma unroll
    for (int i = 0; i < TM; ++i) af[i] = *reinterpret_cast<const bf16x8*>(&S[a_frag + i * 16 * BK + sw]);
  };
  auto compute = [&]() {
    __builtin_amdgcn_s_setprio(1);
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j)
        acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(bfr[j], af[i], acc[i][j], 0, 0, 0);
    __builtin_amdgcn_s_setprio(0);
  };
  auto step = [&](auto up_tag, bf16_t* cur, bf16_t* nxt, int t) {
    constexpr bool UP = decltype(up_tag)::value;
    if constexpr (EARLY) load(up_tag, nxt, t + 1);
    read(cur, 0);
    if constexpr (!EARLY) load(up_tag, nxt, t + 1);
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    pp_barrier();
    compute();
    pp_barrier();
    read(cur, 1);
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    if constexpr (!UP) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    pp_barrier();
    compute();
    if constexpr (UP) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    pp_barrier();
  };
  auto run = [&](auto up_tag) {
    for (int t = 0; t < nk; t += 2) {
      step(up_tag, S0, S1, t);
      if (t + 1 < nk) step(up_tag, S1, S0, t + 1);
    }
  };
  if (upper) {
    load(std::true_type(), S0, 0);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    pp_barrier();
    run(std::true_type());
    pp_barrier();
  } else {
    load(std::false_type(), S0, 0);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    pp_barrier();
    pp_barrier();  // one interval behind
    run(std::false_type());
  }
  __syncthreads();

  // every wave's fragment reads and loads are done: the stages become the staging regions
  const GemmParams e = late_params();
  static_assert(4 * WM * WN <= SZ, "staging space");
  bf16_t* region = (wave < 4 ? S0 : S1) + (wave & 3) * (WM * WN);
  const int64_t mw = m0 + wm * WM, nw = n0 + wn * WN;
  bool done = true;
  switch (e.epi) {
    case EPI_PLAIN: staged_epilogue<EPI_PLAIN, TM, TN, WM, WN>(e, 0, 0, mw, nw, acc, region); break;
    case EPI_BIAS: staged_epilogue<EPI_BIAS, TM, TN, WM, WN>(e, 0, 0, mw, nw, acc, region); break;
    case EPI_BIAS_GELU: staged_epilogue<EPI_BIAS_GELU, TM, TN, WM, WN>(e, 0, 0, mw, nw, acc, region); break;
    case EPI_BIAS_SILU: staged_epilogue<EPI_BIAS_SILU, TM, TN, WM, WN>(e, 0, 0, mw, nw, acc, region); break;
    case EPI_BIAS_RES: staged_epilogue<EPI_BIAS_RES, TM, TN, WM, WN>(e, 0, 0, mw, nw, acc, region); break;
    case EPI_RES: staged_epilogue<EPI_RES, TM, TN, WM, WN>(e, 0, 0, mw, nw, acc, region); break;
    case EPI_GEGLU_GELU: staged_geglu_epilogue<EPI_GEGLU_GELU, TM, TN, WM, WN>(e, 0, 0, mw, nw, acc, region); break;
    case EPI_GEGLU_SILU: staged_geglu_epilogue<EPI_GEGLU_SILU, TM, TN, WM, WN>(e, 0, 0, mw, nw, acc, region); break;
    case EPI_QKV: done = staged_qkv_epilogue<false, TM, TN, WM, WN>(e, mw, nw, acc, region); break;
    case EPI_QKV_BIAS: done = staged_qkv_epilogue<true, TM, TN, WM, WN>(e, mw, nw, acc, region); break;
    default: done = false; break;
  }
  // one call site: also a wave whose QKV slab straddles two parts
  if (!done) mfma_epilogue<bf16_t, TM, TN>(e, 0, 0, mw + fr, nw + 4 * fc, acc);
}

bool gemm_pp_takes(int64_t M, int64_t N, int64_t K, int epi, int cus) {
  // The epilogues that this kernel stages; a K loop that amortises its start (8192 x 8192 x 64 42
  // us against 34, x 256 equal); tiles that fill most of their rounds: at 0.75 of them 8192 x 3072 x
  // 768 59 against 54 us and 8192 x 3072 x 1024 61 against 58, but 6000 x 4096 x 2048 100 against
  // 108; at 0.83 8192 x 5120 x 2048 159 against 176, at 0.875 8192 x 7168 x 512 equal, 8192 x 3584 x
  // 2048 105 against 144.
  if (epi == EPI_GENERIC || K < 256) return false;
  const int64_t tiles = ((M + 255) / 256) * ((N + 255) / 256), rounds = (tiles + cus - 1) / cus;
  const double filled = (double)M * (double)N / (65536.0 * (double)(rounds * cus));
  return filled >= (K >= 2048 ? 0.74 : 0.8);
}

int gemm_pp_launch(tl_ctx* ctx, GemmParams p, int family, double flops, double bytes) {
  p.tiles_m = (int)((p.M + 255) / 256);
  p.tiles_n = (int)((p.N + 255) / 256);
  TL_REQUIRE((int64_t)p.tiles_m * p.tiles_n < 0x7fffffff, "too many tiles");
  const dim3 grid((unsigned)(p.tiles_m * p.tiles_n));
  LaunchScope ls(ctx, family, flops, bytes);
  // far-apart rows miss more caches: loads before the reads (K = 16384 465 -> 433 us; 8192 equal,
  // 4096 113 against 122)
  if (p.K > 8192) gemm_pp_kernel<true><<<grid, 512, 0, ctx->stream>>>(p);
  else gemm_pp_kernel<false><<<grid, 512, 0, ctx->stream>>>(p);
  return ls.finish("gemm_pp");
}

}  // namespace tl
