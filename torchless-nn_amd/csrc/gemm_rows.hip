// gemm_rows_kernel: products with too few output tiles to fill the chip on the tiles of
// gemm.hip: those of a batched decode step (M = 17 .. 128 rows: a stream of the weights), of a
// few short prompts, of a small model. bf16 operands on v_mfma_f32_16x16x32_bf16, fp32 ones on
// v_mfma_f32_16x16x4f32 (as in gemm_mfma_f32_kernel).
//
// What bounds them is the weight stream and the start of a workgroup, not the matrix cores,
// so a workgroup keeps whole K steps of both operands in flight on their way into LDS
// (global_load_lds_dwordx4 as in gemm_dma_kernel: no registers held, a ring of STAGES
// buffers) and K is cut twice to put more loads in flight: WGK waves of a workgroup take
// different K slices (128 bytes of a row) of a stage (their sums meet in LDS), and p.splits workgroups
// take different K ranges of one output tile (fp32 partial sums in the workspace, added in
// order by gemm_rows_reduce_kernel, which runs the epilogue).
#include <algorithm>

#include "gemm_common.hpp"
#include "gemm_rows.hpp"

namespace tl {

// Waits until at most N vector memory operations of this wave are outstanding, N known only
// as a multiple r * L with r <= R (the wait count is an immediate).
template <int L, int R>
__device__ __forceinline__ void stage_sync_upto(int r) {
  if constexpr (R == 0) {
    dma_stage_sync<0>();
  } else {
    if (r >= R) dma_stage_sync<L * R>();
    else stage_sync_upto<L, R - 1>(r);
  }
}

template <typename T> struct Frag { typedef bf16x8 type; };
template <> struct Frag<float> { typedef f32x4 type; };

template <typename TI, typename TO, int BM, int BN, int WGM, int WGN, int WGK, int STAGES>
__global__ __launch_bounds__(64 * WGM * WGN * WGK) void gemm_rows_kernel(GemmParams p, float* part,
                                                                        int splits) {
  constexpr int NW = WGM * WGN * WGK, CH = 16 / sizeof(TI);  // elements of a 16-byte chunk
  constexpr int BK = 8 * CH;                       // a K slice: 8 chunks, 128 bytes per row
  constexpr int WM = BM / WGM, WN = BN / WGN, TM = WM / 16, TN = WN / 16;
  constexpr int SLICE = (BM + BN) * BK;            // elements of one K slice
  constexpr int GA = BM / 8, GS = (BM + BN) / 8;   // 1 KB load groups of A, and of a slice
  constexpr int L = WGK * GS / NW;                 // load groups per wave and stage
  static_assert(WGK * GS % NW == 0 && TM >= 1 && TN >= 1, "bad tile/wave split");
  static_assert(L * (STAGES - 2) <= 63, "vmcnt range");
  static_assert(STAGES * WGK * SLICE * sizeof(TI) <= 160 * 1024, "LDS");
  static_assert((WGK - 1) * WGM * WGN * TM * TN * 1024 <= STAGES * WGK * SLICE * sizeof(TI), "reduction space");
  __shared__ __attribute__((aligned(16))) TI S[STAGES * WGK * SLICE];

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wk = wave / (WGM * WGN), wmn = wave - wk * (WGM * WGN);
  const int wm = wmn / WGN, wn = wmn - wm * WGN;

  // (split, tile) from the block id: each XCD walks a contiguous run, tile fastest
  int tm, tn, split;
  {
    const int ntiles = p.tiles_m * p.tiles_n, total = ntiles * splits;
    const int x = blockIdx.x & 7, local = blockIdx.x >> 3;
    const int c = x * (total >> 3) + min(x, total & 7) + local;
    split = c / ntiles;
    grouped_tile(c - split * ntiles, p, tm, tn);
  }
  const int64_t m0 = (int64_t)tm * BM, n0 = (int64_t)tn * BN;
  // this workgroup's K slices [s0, s0 + ns)
  const int nslices = (int)(p.K / BK);
  const int per = (nslices + splits - 1) / splits;
  const int s0 = min(split * per, nslices), ns = min(per, nslices - s0);

  const TI* Ab = (const TI*)p.A + m0 * p.lda;
  const TI* Bb = (const TI*)p.B + n0 * p.ldb;
  // Load group q of a stage (q = wave * L + j) is group q % GS of slice q / GS: 8 tile rows x
  // 8 chunks, lane l fills row l / 8, slot l % 8 with chunk (l % 8) ^ (row % 8). Rows past M
  // or N are clamped to the last one: computed, never stored.
  uint32_t off[L];
  {
    const int a_last = (int)min((int64_t)BM - 1, p.M - 1 - m0);
    const int b_last = (int)min((int64_t)BN - 1, p.N - 1 - n0);
    const int rin = lane >> 3, c = (lane & 7) ^ rin;
#pragma unroll
    for (int j = 0; j < L; ++j) {
      const int g = (wave * L + j) % GS;
      off[j] = g < GA ? (uint32_t)(min(8 * g + rin, a_last) * p.lda + c * CH)
                      : (uint32_t)(min(8 * (g - GA) + rin, b_last) * p.ldb + c * CH);
    }
  }
  const int nst = (ns + WGK - 1) / WGK;  // stages
  auto issue = [&](int t, int buf) {
    TI* dst = S + buf * (WGK * SLICE);
#pragma unroll
    for (int j = 0; j < L; ++j) {
      const int q = wave * L + j, sl = q / GS, g = q - sl * GS;
      // a slice past the end reads the last one again (in bounds; it is not computed)
      const int64_t k = (int64_t)(s0 + min(t * WGK + sl, ns - 1)) * BK;
      dma_load16((g < GA ? Ab : Bb) + k + off[j], lds_offset(dst + q * (8 * BK)));
    }
  };
  f32x4 acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  const int fr = lane & 15, fc = lane >> 4;
  const int a_frag = wk * SLICE + (wm * WM + fr) * BK;
  const int b_frag = wk * SLICE + BM * BK + (wn * WN + fr) * BK;
#pragma unroll
  for (int t = 0; t < STAGES - 1; ++t)
    if (t < nst) issue(t, t);
  int cur = 0;  // ring position of stage t; stage t + STAGES - 1 goes into the one before it
  for (int t = 0; t < nst; ++t) {
    stage_sync_upto<L, STAGES - 2>(nst - 1 - t);  // later stages may stay in flight
    if (t + STAGES - 1 < nst) issue(t + STAGES - 1, cur == 0 ? STAGES - 1 : cur - 1);
    if (WGK == 1 || t * WGK + wk < ns) {
      const TI* St = S + cur * (WGK * SLICE);
      typename Frag<TI>::type af[2][TM], bfr[2][TN];
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const int sw = ((h * 4 + fc) ^ (fr & 7)) * CH;
#pragma unroll
        for (int i = 0; i < TM; ++i) af[h][i] = *reinterpret_cast<const typename Frag<TI>::type*>(&St[a_frag + i * 16 * BK + sw]);
#pragma unroll
        for (int j = 0; j < TN; ++j) bfr[h][j] = *reinterpret_cast<const typename Frag<TI>::type*>(&St[b_frag + j * 16 * BK + sw]);
      }
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        if constexpr (sizeof(TI) == 2) {
#pragma unroll
          for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int j = 0; j < TN; ++j)
              acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(bfr[h][j], af[h][i], acc[i][j], 0, 0, 0);
        } else {  // element q of every lane's chunk: K indices 4 c + q of the chunks c
#pragma unroll
          for (int q = 0; q < 4; ++q)
#pragma unroll
            for (int i = 0; i < TM; ++i)
#pragma unroll
              for (int j = 0; j < TN; ++j)
                acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(bfr[h][j][q], af[h][i][q], acc[i][j], 0, 0, 0);
        }
      }
      if constexpr (sizeof(TI) == 2) schedule_kstep<TM + TN, TM * TN>();
    }
    cur = cur + 1 == STAGES ? 0 : cur + 1;
  }

  if constexpr (WGK > 1) {  // the K slices' sums: waves wk > 0 leave theirs in LDS
    f32x4* red = reinterpret_cast<f32x4*>(S);
    __syncthreads();  // every wave has read its last stage
    if (wk > 0) {
      f32x4* mine = red + (int64_t)((wk - 1) * (WGM * WGN) + wmn) * (TM * TN * 64) + lane;
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) mine[(i * TN + j) * 64] = acc[i][j];
    }
    __syncthreads();
    if (wk > 0) return;
#pragma unroll
    for (int w = 0; w < WGK - 1; ++w) {
      const f32x4* other = red + (int64_t)(w * (WGM * WGN) + wmn) * (TM * TN * 64) + lane;
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) acc[i][j] += other[(i * TN + j) * 64];
    }
  }
  const int64_t mb = m0 + wm * WM + fr, nb = n0 + wn * WN + 4 * fc;
  if (splits > 1) {  // part[split][row][column], columns padded to whole tiles
    const int64_t ld = (int64_t)p.tiles_n * BN;
    float* out = part + ((int64_t)split * p.M + mb) * ld + nb;
#pragma unroll
    for (int i = 0; i < TM; ++i) {
      if (mb + 16 * i >= p.M) continue;
#pragma unroll
      for (int j = 0; j < TN; ++j) *reinterpret_cast<f32x4*>(out + (int64_t)16 * i * ld + 16 * j) = acc[i][j];
    }
    return;
  }
  const GemmParams e = late_params();
  mfma_epilogue<TO, TM, TN, TI>(e, 0, 0, mb, nb, acc);
}

// Sums the splits' partials of 4 consecutive columns of one row in order, then the epilogue.
template <typename TI, typename TO>
__global__ __launch_bounds__(256) void gemm_rows_reduce_kernel(GemmParams p, const float* part,
                                                               int splits, int64_t ld) {
  const int64_t n0 = ((int64_t)blockIdx.y * 256 + threadIdx.x) * 4, m = blockIdx.x;
  if (n0 >= p.N) return;
  const float* src = part + m * ld + n0;
  f32x4 t = *reinterpret_cast<const f32x4*>(src);
  for (int s = 1; s < splits; ++s) t += *reinterpret_cast<const f32x4*>(src + (int64_t)s * p.M * ld);
  float v[4] = {t[0], t[1], t[2], t[3]};
  epilogue4<TI, TO>(p, 0, 0, m, n0, v);
}

// The tiles, with what they cost on an MI355X: `start` us from launch to the first stage, then
// `stage1` / `stage2` us per stage with one / two workgroups per CU. Fitted to 280 bf16 (M = 17
// .. 3500, N 256 .. 256000, K 256 .. 16384) and 370 fp32 products (M = 1 .. 33000, N 65 ..
// 50257, K 128 .. 4096), each timed on 2 to 20 (tile, splits) pairs: the pair that the model
// picks takes on average 0.8% (bf16) and 0.3% (fp32, gemm_split.hip's pairs included) more than
// the best one. 128-column tiles stay behind the split kernel's in fp32.
struct RowsTile {
  int bm, bn, wgk, per_cu;
  float start, stage1, stage2;
  float start32, stage1_32, stage2_32;
};
static const RowsTile kRowsTiles[] = {
    {32, 32, 4, 1, 0.3f, 0.50f, 0.60f, 0.2f, 0.91f, 1.0f},
    {32, 64, 2, 2, 0.35f, 0.48f, 0.86f, 0.35f, 0.9f, 1.3f},
    {64, 64, 1, 2, 0.45f, 0.25f, 0.45f, 0.4f, 0.55f, 1.08f},
    {32, 128, 1, 2, 0.4f, 0.50f, 0.56f, 0, 0, 0},
    {64, 128, 1, 2, 0.5f, 0.60f, 0.72f, 0, 0, 0},
    {128, 128, 1, 2, 0.85f, 0.80f, 0.97f, 0, 0, 0},
};
constexpr int kNumRowsTiles = sizeof(kRowsTiles) / sizeof(kRowsTiles[0]), kNumRowsTiles32 = 3;

template <typename TI, typename TO>
static void launch_rows(int tile, dim3 grid, hipStream_t st, const GemmParams& p, float* part, int s) {
  switch (tile) {
    case 0: gemm_rows_kernel<TI, TO, 32, 32, 1, 1, 4, 4><<<grid, 256, 0, st>>>(p, part, s); return;
    case 1: gemm_rows_kernel<TI, TO, 32, 64, 1, 2, 2, 3><<<grid, 256, 0, st>>>(p, part, s); return;
    case 2: gemm_rows_kernel<TI, TO, 64, 64, 2, 2, 1, 5><<<grid, 256, 0, st>>>(p, part, s); return;
  }
  if constexpr (sizeof(TI) == 2) {
    switch (tile) {
      case 3: gemm_rows_kernel<TI, TO, 32, 128, 1, 4, 1, 4><<<grid, 256, 0, st>>>(p, part, s); return;
      case 4: gemm_rows_kernel<TI, TO, 64, 128, 1, 4, 1, 3><<<grid, 256, 0, st>>>(p, part, s); return;
      default: gemm_rows_kernel<TI, TO, 128, 128, 2, 2, 1, 2><<<grid, 256, 0, st>>>(p, part, s); return;
    }
  }
}

static inline int64_t ceil_div(int64_t a, int64_t b) { return (a + b - 1) / b; }

// The cheapest pair among the first `ntiles` tiles by modelled time (us, without what all choices
// share). Up to 50 pairs are priced on every call, in 32-bit arithmetic: about 1 us of host time.
static RowsPlan rows_best(int64_t M, int64_t N, int64_t K, int elem, int ntiles, int cus) {
  RowsPlan best;
  const uint32_t nslices = (uint32_t)(K / (128 / elem));
  const float sums = (float)M * (float)N * (8 / 2e6f);  // partial sums written and read, per split
  for (int i = 0; i < ntiles; ++i) {
    const RowsTile& t = kRowsTiles[i];
    if (t.bm > 32 && t.bm >= 2 * M) continue;  // half padding
    const uint64_t tiles64 = (uint64_t)(((uint32_t)M + t.bm - 1) / t.bm) * (((uint32_t)N + t.bn - 1) / t.bn);
    if (tiles64 > (1 << 24)) continue;
    const uint32_t tiles = (uint32_t)tiles64, slots = (uint32_t)(t.per_cu * cus);
    const float start = elem == 2 ? t.start : t.start32;
    const float stage1 = elem == 2 ? t.stage1 : t.stage1_32, stage2 = elem == 2 ? t.stage2 : t.stage2_32;
    for (const uint32_t s : {1u, 2u, 3u, 4u, 5u, 6u, 8u, 10u, 12u, 16u}) {
      // each part keeps at least three slices, and the parts fit four workgroups per CU
      if (s > 1 && (nslices < 3 * s || tiles * s > 4u * (uint32_t)cus)) break;
      const float stages = (float)(((nslices + s - 1) / s + t.wgk - 1) / t.wgk);
      const float one = start + stages * stage1, two = start + stages * stage2;
      const uint32_t full = tiles * s / slots, rest = tiles * s - full * slots;
      float us = (float)full * (t.per_cu == 1 ? one : two);
      if (rest) us += rest <= (uint32_t)cus ? one : two;
      if (s > 1) us += 2.0f + (float)s * sums;  // and a second launch, on the host as well
      if (best.tile < 0 || us < best.us) {
        best.tile = i;
        best.splits = (int)s;
        best.us = us;
      }
    }
  }
  return best;
}

RowsPlan gemm_rows_plan(int64_t M, int64_t N, int64_t K, int cus, bool can_stream) {
  // M <= 16: the weight-streaming kernels of gemm.hip start faster (3 to 30% on K <= 2048), but
  // gemm_skinny_kernel loads and multiplies the activation rows again for every 16 columns, which
  // costs more the more rows there are. Over 32768 to 256000 columns with weights that come from
  // HBM (us, there / here): 1 x 50257 x 256 12.9 / 8.6, 4 x 50257 x 768 19.5 / 17.4, 16 x 50257 x 768
  // 25.1 / 18.3, 4 x 256000 x 1024 98.9 / 93.3, 16 x 256000 x 1024 143 / 99; but 1 x 256000 x 1024 85.3 /
  // 89.4, 1 x 50257 x 1536 28.6 / 31.7. On K > 768 four rows break even over seven widths (0.93 to 1.09).
  // gemm_skinny_stream_kernel (K % 2048 == 0) keeps the rows in registers and stays ahead: 4 x
  // 50257 x 2048 40.4 / 44.9, 4 x 65536 x 2048 49 / 59, 4 x 256000 x 2048 173 / 178, 16 x 32768 x 2048
  // 28 / 31, 4 x 65536 x 4096 102 / 110 (K = 4096 beyond 150000 columns: 227 / 216). Its K parts need
  // a workspace, which this kernel can do without.
  if (M <= 16) {
    const bool here = N >= 32768 && (K % 2048 == 0 ? !can_stream : K <= 768 || M >= 4);
    return here ? rows_best(M, N, K, 2, kNumRowsTiles, cus) : RowsPlan();
  }
  // Products that fill the chip on the tiles of gemm.hip stay there (at 2331 x 2304 x 768 14.9
  // us against 18.8 here), with two exceptions. M <= 64, or <= 128 over many columns, is a
  // stream of the weights, and 256-row tiles only load padding with it (48 x 32768 x 2048 42.4
  // -> 35.4 us, 20 x 256000 x 2048 276 -> 187, 128 x 50257 x 768 33.9 -> 28.0; 128 x 32768 x
  // 2048, one tile per CU either way, 43.2 against 46.8). A long K with up to 1.25 tiles of 128 x
  // 128 per CU gains from the split (1500 x 2048 x 16384 201 -> 133 us, 2331 rows 204 -> 189;
  // 3500 rows, 1.75 tiles per CU, 216 against 239). What does not fill it, and ran on 64-row
  // register-prefetch tiles before, gains throughout (226 products, 1.08 to 11.9 times as fast,
  // median 1.76: 24 x 2048 x 16384 237 -> 20.5 us, 400 x 768 x 3072 35 -> 13).
  const int64_t t96 = ceil_div(M, 128) * ceil_div(N, 96), t96w = ceil_div(M, 256) * ceil_div(N, 96);
  const int64_t t128 = ceil_div(M, 128) * ceil_div(N, 128);
  const bool fills = t96 >= cus || (K >= 256 && t96w >= cus);
  const bool stream = M <= 64 || (M <= 128 && t128 * 2 >= 3LL * cus);
  const bool long_k = K >= 4096 && t128 * 4 <= 5LL * cus;
  if (fills && !stream && !long_k) return RowsPlan();
  return rows_best(M, N, K, 2, kNumRowsTiles, cus);
}

RowsPlan gemm_rows_plan_f32(int64_t M, int64_t N, int64_t K, int cus) {
  return rows_best(M, N, K, 4, kNumRowsTiles32, cus);
}

template <typename TI, typename TO>
static void launch_rows_all(const RowsPlan& plan, dim3 grid, hipStream_t st, const GemmParams& p,
                            float* part, int64_t ld) {
  launch_rows<TI, TO>(plan.tile, grid, st, p, part, plan.splits);
  if (plan.splits > 1) {
    const dim3 rgrid((unsigned)p.M, (unsigned)((p.N + 1023) / 1024));
    gemm_rows_reduce_kernel<TI, TO><<<rgrid, 256, 0, st>>>(p, part, plan.splits, ld);
  }
}

int gemm_rows_launch(tl_ctx* ctx, GemmParams p, RowsPlan plan, bool f32in, bool f32out, int family,
                     double flops, double bytes) {
  const RowsTile& t = kRowsTiles[plan.tile];
  p.tiles_m = (int)((p.M + t.bm - 1) / t.bm);
  p.tiles_n = (int)((p.N + t.bn - 1) / t.bn);
  const int64_t ld = (int64_t)p.tiles_n * t.bn;
  float* part = nullptr;
  if (plan.splits > 1) {  // without room for the partial sums one workgroup takes all of K
    part = (float*)try_workspace(ctx, (size_t)plan.splits * p.M * ld * sizeof(float));
    if (!part) plan.splits = 1;
  }
  const dim3 grid((unsigned)((int64_t)p.tiles_m * p.tiles_n * plan.splits));
  LaunchScope ls(ctx, family, flops, bytes);
  if (f32in && f32out) launch_rows_all<float, float>(plan, grid, ctx->stream, p, part, ld);
  else if (f32in) launch_rows_all<float, bf16_t>(plan, grid, ctx->stream, p, part, ld);
  else if (f32out) launch_rows_all<bf16_t, float>(plan, grid, ctx->stream, p, part, ld);
  else launch_rows_all<bf16_t, bf16_t>(plan, grid, ctx->stream, p, part, ld);
  return ls.finish("gemm_rows");
}

}  // namespace tl
