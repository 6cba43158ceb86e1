// gemm_split_kernel: large fp32 products on the bf16 matrix cores. The fp32 MFMA peaks at 157
// TFLOP/s, the bf16 one at 2.5 PFLOP/s, so six bf16 products per fp32 product have 2.6 times
// the room.
//
// Every operand element is split into three bf16 pieces and the six products above 2^-24 are
// taken (fp32_pieces.hpp), with fewer fp32 roundings than the fp32 MFMA's (6 accumulating
// instructions per 32 of K instead of 8).
//
// What the pieces cannot represent is recomputed: an infinity, a NaN or a value that rounds past
// bf16's largest gives a NaN or infinite sum, and parts of tiny elements that are lost matter only
// in sums that are small beside the tile's largest element (fp32_pieces.hpp). A wave that holds a
// nonzero sum outside [least, inf), least = max(2^-60, K 2^-96 largest), redoes its block with the
// fp32 MFMA straight from memory, and so does one that holds a 0 whose row or column has an element
// below 2^-63 (zeros_doubtful). Such results are what gemm_mfma_f32_kernel gives.
//
// Layout: K steps of 32; the fp32 elements of the next step are loaded into registers, split on
// the vector ALUs and written as three bf16 planes [rows][32] to LDS (16-byte chunks, XOR-swizzled
// by row / 2, so that the writes and the fragment reads meet no bank conflicts). Two forms: 256x128
// with 8 waves of 64x64 and two LDS buffers, where a step's splitting (132 vector instructions per
// wave) is scheduled among the 96 MFMAs of the step before it, and 128x64 with 4 waves of 64x32 and
// one buffer, three workgroups per CU, whose phases overlap each other's. Once the chip is full the
// matrix cores are busy 0.42 to 0.46 of the time and each of the two waves per SIMD issues vector
// instructions for 0.22 of it; neither alone bounds it: 8192 x 50257 x 768 5801 ->
// 3262 us (194 TFLOP/s of fp32 products, 1.16 PFLOP/s on the matrix cores), 4000 x 3072 x 768 174 ->
// 107, 4000 x 768 x 3072 230 -> 108 us; error against 64 bits 4.2e-7 where the fp32 MFMA's is
// 5.0e-7 (1024 x 50257 x 768; 0.78 to 0.85 of it over 10007 to 50257 columns, K 256 .. 768). The
// largest element and the look at the sums cost nothing that shows (before and after: 4000 x 3072 x
// 768 123 and 123 us, 4000 x 768 x 3072 126 and 125, 2048 x 2048 x 256 23.6 and 22.3).
#include <algorithm>

#include "fp32_pieces.hpp"
#include "gemm_split.hpp"

namespace tl {

// Whether one of a wave's sums that are 0 belongs to a row of A or of B with a tiny element: rows a0 + r
// (r < 16 TM, clamped to a_last) of A, b0 + c of B, K elements each. A row of A that is all zeros
// has sums of 0 whatever the columns hold. Wave-uniform.
template <int TM, int TN>
__device__ __forceinline__ bool zeros_doubtful(const f32x4 (&acc)[TM][TN], const float* A, int64_t lda, int a0, int a_last,
                                               const float* B, int64_t ldb, int b0, int b_last, int K) {
  const int lane = threadIdx.x & 63, fr = lane & 15;
  auto scan = [&](const float* row, bool& tiny) {  // whether the row has a nonzero element
    bool some = false;
    for (int k = lane * 4; k < K; k += 256) {
      const f32x4 x = *reinterpret_cast<const f32x4*>(row + k);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        some |= x[e] != 0.f;
        tiny |= pieces_tiny(x[e]);
      }
    }
    tiny = __any(tiny);
    return __any(some);
  };
  bool tiny = false;
  uint64_t rows = 0, cols = 0;  // those with sums of 0
#pragma unroll
  for (int i = 0; i < TM; ++i) {
    bool z = false;
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int q = 0; q < 4; ++q) z |= acc[i][j][q] == 0.f;
    uint64_t b = __ballot(z);
    b |= b >> 32;
    b |= b >> 16;
    rows |= (b & 0xffff) << (16 * i);
  }
  for (uint64_t left = rows; left; left &= left - 1) {
    const int r = __builtin_ctzll(left);
    if (!scan(A + (int64_t)min(a0 + r, a_last) * lda, tiny)) rows &= ~(1ull << r);
    if (tiny) return true;
  }
  if (!rows) return false;
#pragma unroll
  for (int j = 0; j < TN; ++j)
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      bool z = false;
#pragma unroll
      for (int i = 0; i < TM; ++i) z |= acc[i][j][q] == 0.f && (rows >> (16 * i + fr) & 1);
      const uint64_t b = __ballot(z);
#pragma unroll
      for (int g = 0; g < 4; ++g) cols |= (uint64_t)((b >> (16 * g) & 0xffff) != 0) << (16 * j + 4 * g + q);
    }
  for (; cols; cols &= cols - 1) {
    scan(B + (int64_t)min(b0 + __builtin_ctzll(cols), b_last) * ldb, tiny);
    if (tiny) return true;
  }
  return false;
}

template <typename TO, int BM, int BN, int WGM, int WGN, int NBUF>
__global__ __launch_bounds__(64 * WGM * WGN) void gemm_split_kernel(GemmParams p, float* part, int full, int splits) {
  constexpr int NT = 64 * WGM * WGN, BK = 32;
  constexpr int WM = BM / WGM, WN = BN / WGN, TM = WM / 16, TN = WN / 16;
  constexpr int ROWS = BM + BN, PLANE = ROWS * BK;  // elements of one bf16 plane
  constexpr int CPT = ROWS * 4 / NT;                // 8-element chunks per thread and step
  static_assert(ROWS * 4 % NT == 0 && BM * 4 % NT == 0 && TM >= 1 && TN >= 1, "bad tile/thread split");
  static_assert(NBUF * 3 * PLANE * 2 <= 160 * 1024, "LDS");
  __shared__ __attribute__((aligned(16))) bf16_t S[NBUF][3 * PLANE];
  __shared__ float wave_most[WGM * WGN];

  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wm = wave / WGN, wn = wave - wm * WGN;
  // The first `full` tiles of the order take one workgroup each, the others `splits`, with a
  // part of K each; within both kinds every XCD walks a contiguous run.
  auto xcd_run = [](int i, int total) {
    const int x = i & 7;
    return x * (total >> 3) + min(x, total & 7) + (i >> 3);
  };
  const int ntiles = p.tiles_m * p.tiles_n, nk_all = (int)(p.K / BK);
  const bool whole = (int)blockIdx.x < full;
  int tile, k_begin = 0, nk = nk_all;
  int64_t piece = 0;  // of the partial sums
  if (whole) {
    tile = xcd_run((int)blockIdx.x, full);
  } else {
    const int rest = ntiles - full;
    const int u = xcd_run((int)blockIdx.x - full, rest * splits), s = u / rest;
    tile = full + (u - s * rest);
    piece = u;
    const int per = (nk_all + splits - 1) / splits;
    k_begin = s * per;  // the host takes care that no part is empty
    nk = min(per, nk_all - k_begin);
  }
  int tm, tn;
  grouped_tile(tile, p, tm, tn);
  const int64_t m0 = (int64_t)tm * BM, n0 = (int64_t)tn * BN;
  k_begin *= BK;
  const int K = nk * BK;
  const float* Ab = (const float*)p.A + m0 * p.lda + k_begin;
  const float* Bb = (const float*)p.B + n0 * p.ldb + k_begin;

  // Chunk q = i * NT + tid of a step: row q / 4 (rows of A, then of B), columns 8 (q % 4) ..;
  // rows past M or N are clamped to the last one (computed, never stored).
  uint32_t off[CPT];
  const int lc = tid & 3;
  {
    const int a_last = (int)min((int64_t)BM - 1, p.M - 1 - m0);
    const int b_last = (int)min((int64_t)BN - 1, p.N - 1 - n0);
#pragma unroll
    for (int i = 0; i < CPT; ++i) {
      const int r = (i * NT + tid) >> 2;
      off[i] = i < BM * 4 / NT ? (uint32_t)(min(r, a_last) * p.lda + lc * 8)
                               : (uint32_t)(min(r - BM, b_last) * p.ldb + lc * 8);
    }
  }
  float raw[CPT][8];
  auto load = [&](int k0) {
#pragma unroll
    for (int i = 0; i < CPT; ++i) {
      const float* src = (i < BM * 4 / NT ? Ab : Bb) + off[i] + k0;
      const f32x4 u = *reinterpret_cast<const f32x4*>(src);
      const f32x4 v = *reinterpret_cast<const f32x4*>(src + 4);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        raw[i][e] = u[e];
        raw[i][4 + e] = v[e];
      }
    }
  };
  // every pass of chunks shares one swizzled slot: NT / 4 rows are a multiple of 8
  const int slot = (tid >> 2) * BK + ((lc ^ ((tid >> 3) & 3)) << 3);
  float most = 0.f;  // largest magnitude this thread has split
  auto store = [&](bf16_t* B) {
#pragma unroll
    for (int i = 0; i < CPT; ++i) {
      uint4 p1, p2, p3;
      split8(raw[i], p1, p2, p3, most);
      bf16_t* dst = B + slot + i * (NT / 4) * BK;
      *reinterpret_cast<uint4*>(dst) = p1;
      *reinterpret_cast<uint4*>(dst + PLANE) = p2;
      *reinterpret_cast<uint4*>(dst + 2 * PLANE) = p3;
    }
  };

  f32x4 acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  const int fr = lane & 15, fc = lane >> 4;
  const int sw = (fc ^ ((fr >> 1) & 3)) << 3;
  const int a_frag = (wm * WM + fr) * BK + sw, b_frag = (BM + wn * WN + fr) * BK + sw;
  auto compute = [&](const bf16_t* B) {
    bf16x8 b[3][TN];
#pragma unroll
    for (int pl = 0; pl < 3; ++pl)
#pragma unroll
      for (int j = 0; j < TN; ++j)
        b[pl][j] = *reinterpret_cast<const bf16x8*>(B + pl * PLANE + b_frag + j * 16 * BK);
#pragma unroll
    for (int i = 0; i < TM; ++i) {
      bf16x8 a[3];
#pragma unroll
      for (int pl = 0; pl < 3; ++pl)
        a[pl] = *reinterpret_cast<const bf16x8*>(B + pl * PLANE + a_frag + i * 16 * BK);
      // smallest products first; one row of fragments at a time (pairs of rows, for more sums
      // between two products of one, took 30% longer on 4000 x 2304 x 768)
#pragma unroll
      for (int t = 0; t < 6; ++t)
#pragma unroll
        for (int j = 0; j < TN; ++j)
          acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(b[kPieceB[t]][j], a[kPieceA[t]], acc[i][j], 0, 0, 0);
    }
  };

  load(0);
  if constexpr (NBUF == 2) {
    store(S[0]);
    load(min(1, nk - 1) * BK);
    __syncthreads();
    for (int t = 0; t < nk; ++t) {
      // the last step stores and loads its own elements again: one basic block per step
      compute(S[t & 1]);
      store(S[(t & 1) ^ 1]);
      load(min(t + 2, nk - 1) * BK);
      __syncthreads();
    }
  } else {
    for (int t = 0; t < nk; ++t) {
      store(S[0]);
      load(min(t + 1, nk - 1) * BK);
      __syncthreads();
      compute(S[0]);
      __syncthreads();
    }
  }

  const int64_t mb = m0 + wm * WM + fr, nb = n0 + wn * WN;
  {
    most = wave_max(most);
    if (lane == 0) wave_most[wave] = most;
    __syncthreads();
#pragma unroll
    for (int w = 0; w < WGM * WGN; ++w) most = fmaxf(most, wave_most[w]);
    const float least = pieces_least(most, K);
    bool look = false, bad = false;
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j)
#pragma unroll
        for (int q = 0; q < 4; ++q) look = look || pieces_doubtful(acc[i][j][q], least);
    if (__any(look)) {
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
          for (int q = 0; q < 4; ++q) bad = bad || (pieces_doubtful(acc[i][j][q], least) && acc[i][j][q] != 0.f);
      if (!__any(bad))
        bad = zeros_doubtful<TM, TN>(acc, Ab, p.lda, wm * WM, (int)min((int64_t)BM, p.M - m0) - 1, Bb, p.ldb,
                                     wn * WN, (int)min((int64_t)BN, p.N - n0) - 1, K);
    }
    if (__any(bad)) {  // this wave's block again on the fp32 matrix cores (see above)
      const float* Ar[TM];
      const float* Br[TN];
#pragma unroll
      for (int i = 0; i < TM; ++i) Ar[i] = Ab + (min(mb + 16 * i, p.M - 1) - m0) * p.lda + fc;
#pragma unroll
      for (int j = 0; j < TN; ++j) Br[j] = Bb + (min(nb + 16 * j + fr, p.N - 1) - n0) * p.ldb + fc;
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll 1
      for (int k = 0; k < K; k += 4) {
        float a[TM], b[TN];
#pragma unroll
        for (int i = 0; i < TM; ++i) a[i] = Ar[i][k];
#pragma unroll
        for (int j = 0; j < TN; ++j) b[j] = Br[j][k];
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
          for (int j = 0; j < TN; ++j)
            acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(b[j], a[i], acc[i][j], 0, 0, 0);
      }
    }
  }
  if (!whole) {  // part[piece][row][column], rows and columns of the whole tile
    float* out = part + (piece * BM + wm * WM + fr) * BN + wn * WN + 4 * fc;
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j) *reinterpret_cast<f32x4*>(out + 16 * i * BN + 16 * j) = acc[i][j];
    return;
  }
  const GemmParams e = late_params();
  mfma_epilogue<TO, TM, TN, float>(e, 0, 0, mb, nb + 4 * fc, acc);
}

// Adds the `splits` partial sums of each tile from `full` on, in order, then the epilogue: one
// thread per 4 columns of a row.
template <typename TO, int BM, int BN>
__global__ __launch_bounds__(256) void gemm_split_reduce_kernel(GemmParams p, const float* part,
                                                                int full, int splits) {
  const int at = ((int)blockIdx.y * 256 + (int)threadIdx.x) * 4, r = at / BN, c = at - r * BN;
  const int rest = p.tiles_m * p.tiles_n - full;
  int tm, tn;
  grouped_tile(full + (int)blockIdx.x, p, tm, tn);
  const int64_t m = (int64_t)tm * BM + r, n0 = (int64_t)tn * BN + c;
  if (m >= p.M || n0 >= p.N) return;
  const float* src = part + (int64_t)blockIdx.x * (BM * BN) + at;
  f32x4 t = *reinterpret_cast<const f32x4*>(src);
  for (int s = 1; s < splits; ++s) t += *reinterpret_cast<const f32x4*>(src + (int64_t)s * rest * (BM * BN));
  float v[4] = {t[0], t[1], t[2], t[3]};
  epilogue4<float, TO>(p, 0, 0, m, n0, v);
}

// The tiles and what they cost on an MI355X: `start` us, then step[k - 1] us per 32 of K with k
// workgroups per CU (fitted with gemm_rows.hip's fp32 ones to 370 products).
struct SplitTile {
  int bm, bn, per_cu;
  float start, step[3];
};
static const SplitTile kSplitTiles[] = {{256, 128, 1, 2.3f, {2.06f, 0, 0}}, {128, 64, 3, 1.64f, {1.0f, 1.4f, 2.09f}}};

template <typename TO, int BM, int BN, int WGM, int WGN, int NBUF>
static void launch_split_tile(dim3 grid, hipStream_t st, const GemmParams& p, float* part, const SplitPlan& plan) {
  gemm_split_kernel<TO, BM, BN, WGM, WGN, NBUF><<<grid, 64 * WGM * WGN, 0, st>>>(p, part, plan.full, plan.splits);
  const int rest = p.tiles_m * p.tiles_n - plan.full;
  if (rest > 0)
    gemm_split_reduce_kernel<TO, BM, BN><<<dim3((unsigned)rest, BM * BN / 1024), 256, 0, st>>>(p, part, plan.full, plan.splits);
}

template <typename TO>
static void launch_split(const SplitPlan& plan, dim3 grid, hipStream_t st, const GemmParams& p, float* part) {
  if (plan.tile == 0) launch_split_tile<TO, 256, 128, 4, 2, 2>(grid, st, p, part, plan);
  else launch_split_tile<TO, 128, 64, 2, 2, 1>(grid, st, p, part, plan);
}

SplitPlan gemm_split_plan(int64_t M, int64_t N, int64_t K, int cus) {
  SplitPlan best;
  const uint32_t nk = (uint32_t)(K / 32);
  for (int i = 0; i < 2; ++i) {
    const SplitTile& t = kSplitTiles[i];
    const uint64_t tiles64 = (uint64_t)(((uint32_t)M + t.bm - 1) / t.bm) * (((uint32_t)N + t.bn - 1) / t.bn);
    if (t.bm >= 4 * M || tiles64 > (1 << 24)) continue;
    const uint32_t tiles = (uint32_t)tiles64, slots = (uint32_t)(t.per_cu * cus);
    auto round = [&](uint32_t wgs, uint32_t steps) {  // one round of at most `slots` workgroups
      return wgs ? t.start + (float)steps * t.step[(wgs - 1) / (uint32_t)cus] : 0.f;
    };
    const uint32_t rounds = tiles / slots, rest = tiles - rounds * slots;
    // What the whole rounds leave would hold the chip for a round however few tiles it is: its
    // tiles may be split over K, for a reduce launch and their partial sums written and read
    // (4000 x 2304 x 768, 288 tiles of 256x128 on 256 CUs: 112.6 us whole, 83.9 with the last
    // 32 in eight parts each; 2331 x 768 x 3072, 60 tiles: 178 whole, 69.9 in four parts).
    for (const uint32_t s : {1u, 2u, 3u, 4u, 6u, 8u}) {
      if (s > 1 && (rest == 0 || nk < 3 * s || rest * s * 5 > slots * 11)) break;
      const uint32_t per = (nk + s - 1) / s, pieces = rest * s, more = pieces / slots;
      float us = (float)rounds * round(slots, nk) + (float)more * round(slots, per) +
                 round(pieces - more * slots, per);
      if (s > 1) us += 3.0f + (float)(pieces * (uint32_t)(t.bm * t.bn / 1024)) * (8192 / 4.9e6f);
      if (best.tile < 0 || us < best.us) {
        best.tile = i;
        best.splits = (int)((nk + per - 1) / per);
        best.full = (int)(best.splits == 1 ? tiles : tiles - rest);
        best.us = us;
      }
    }
  }
  return best;
}

int gemm_split_launch(tl_ctx* ctx, GemmParams p, SplitPlan plan, bool f32out, int family,
                      double flops, double bytes) {
  const SplitTile& t = kSplitTiles[plan.tile];
  p.tiles_m = (int)((p.M + t.bm - 1) / t.bm);
  p.tiles_n = (int)((p.N + t.bn - 1) / t.bn);
  const int64_t tiles = (int64_t)p.tiles_m * p.tiles_n;
  int64_t rest = tiles - plan.full;
  float* part = nullptr;
  if (rest > 0) {  // without room for the partial sums every tile takes one workgroup
    part = (float*)try_workspace(ctx, (size_t)(rest * plan.splits) * t.bm * t.bn * sizeof(float));
    if (!part) {
      plan.full = (int)tiles;
      plan.splits = 1;
      rest = 0;
    }
  }
  const dim3 grid((unsigned)(plan.full + rest * plan.splits));
  LaunchScope ls(ctx, family, flops, bytes);
  if (f32out) launch_split<float>(plan, grid, ctx->stream, p, part);
  else launch_split<bf16_t>(plan, grid, ctx->stream, p, part);
  return ls.finish("gemm_split");
}

}  // namespace tl
