// The LDS-staged bf16 epilogues of the tiled GEMM kernels (gemm.hip, gemm_pp.hip).
#pragma once

#include "gemm_common.hpp"

namespace tl {

// bf16 epilogue through LDS. Each wave applies its epilogue kind to its WM x WN results in
// fp32 (bias, then activation, then residual, as mfma_epilogue does), rounds them once to
// bf16 and writes them to its own LDS region; it then reads them back as 16-byte row pieces
// (U = WN / 8 per row), so each global store instruction writes whole row segments of
// 64 / U rows instead of 32-byte pieces of 16 rows (4x fewer cache lines touched per byte:
// the store issue time per tile drops about 4x). Piece u of row r sits at slot (u + r) % U,
// which spreads the fragment writes over the LDS banks. Only this wave touches its region
// and the LDS operations of one wave complete in order, so the reads need no barrier.
template <int KIND>
struct EpiTraits {
  static constexpr bool BIAS = KIND == EPI_BIAS || KIND == EPI_BIAS_GELU || KIND == EPI_BIAS_SILU ||
                               KIND == EPI_BIAS_RES;
  static constexpr bool RES = KIND == EPI_BIAS_RES || KIND == EPI_RES;
};

// The bias values of a lane's fragment columns nw + 16 j + 4 (lane / 16) + q (0 past N).
template <int KIND, int TN>
__device__ __forceinline__ void load_epi_bias(const GemmParams& e, int64_t nw,
                                              float (&bias)[EpiTraits<KIND>::BIAS ? TN : 1][4]) {
  if constexpr (EpiTraits<KIND>::BIAS) {
    const int fc = (threadIdx.x & 63) >> 4;
#pragma unroll
    for (int j = 0; j < TN; ++j) {
      const int64_t n = nw + 16 * j + 4 * fc;
#pragma unroll
      for (int q = 0; q < 4; ++q) bias[j][q] = bias_at(e, n + q);
    }
  }
}

// Applies epilogue KIND to the fragment rows i = I0 .. I0 + NI - 1 of a wave's accumulators
// (block rows 16 I0 .. 16 (I0 + NI) - 1, starting at global row mw + 16 I0) and writes them,
// rounded once to bf16, to the region as 16-byte row pieces: piece u of staged row r at slot
// (r * U + (u + r) % U), U = WN / 8 (the rotation spreads the fragment writes over the LDS
// banks).
template <int KIND, int TM, int TN, int WN, int I0, int NI>
__device__ __forceinline__ void stage_rows(const GemmParams& e, const bf16_t* rz, int64_t mw,
                                           int64_t nw, f32x4 (&acc)[TM][TN],
                                           const float (&bias)[EpiTraits<KIND>::BIAS ? TN : 1][4],
                                           uint8_t* reg) {
  constexpr bool BIAS = EpiTraits<KIND>::BIAS, RES = EpiTraits<KIND>::RES;
  constexpr int U = WN / 8;
  const int lane = threadIdx.x & 63, fr = lane & 15, fc = lane >> 4;
  // All residual pieces of these rows are requested before any is used (one memory round
  // trip, not one per fragment). Rows past M and columns past N are computed and staged but
  // never stored, so their reads are clamped to the last row and to column N - 4 (N % 4 == 0
  // on this path) and their values do not matter.
  uint2 rv[RES ? NI : 1][RES ? TN : 1];
  if constexpr (RES) {
#pragma unroll
    for (int ii = 0; ii < NI; ++ii) {
      const int64_t m = mw + 16 * (I0 + ii) + fr;
      const bf16_t* rrow = rz + (m < e.M ? m : e.M - 1) * e.ldr;
#pragma unroll
      for (int j = 0; j < TN; ++j) {
        const int64_t n = nw + 16 * j + 4 * fc;
        rv[ii][j] = gload8(rrow + (n < e.N ? n : e.N - 4));
      }
    }
  }
#pragma unroll
  for (int ii = 0; ii < NI; ++ii) {
    const int i = I0 + ii, r = 16 * ii + fr;
#pragma unroll
    for (int j = 0; j < TN; ++j) {
      float v[4] = {acc[i][j][0], acc[i][j][1], acc[i][j][2], acc[i][j][3]};
      if (BIAS) {
#pragma unroll
        for (int q = 0; q < 4; ++q) v[q] = v[q] + bias[BIAS ? j : 0][q];
      }
      if (KIND == EPI_BIAS_GELU) {
#pragma unroll
        for (int q = 0; q < 4; ++q) v[q] = gelu_tanh(v[q]);
      }
      if (KIND == EPI_BIAS_SILU) {
#pragma unroll
        for (int q = 0; q < 4; ++q) v[q] = silu_tanh(v[q]);
      }
      if constexpr (RES) {
        const uint2 w = rv[ii][j];
        v[0] = v[0] + __uint_as_float(w.x << 16);
        v[1] = v[1] + __uint_as_float(w.x & 0xffff0000u);
        v[2] = v[2] + __uint_as_float(w.y << 16);
        v[3] = v[3] + __uint_as_float(w.y & 0xffff0000u);
      }
      uint2 w;
      w.x = (uint32_t)f2bf(v[0]) | ((uint32_t)f2bf(v[1]) << 16);
      w.y = (uint32_t)f2bf(v[2]) | ((uint32_t)f2bf(v[3]) << 16);
      const int u = 2 * j + (fc >> 1);
      *reinterpret_cast<uint2*>(reg + (r * U + (u + r) % U) * 16 + (fc & 1) * 8) = w;
    }
  }
}

// bf16 epilogue through LDS. Each wave applies its epilogue kind to its WM x WN results in
// fp32 (bias, then activation, then residual, as mfma_epilogue does), stages them in its own
// LDS region (stage_rows) and reads them back as 16-byte row pieces, so each global store
// instruction writes whole row segments of 64 / U rows instead of 32-byte pieces of 16 rows
// (4x fewer cache lines touched per byte: the store issue time per tile drops about 4x).
// Only this wave touches its region and the LDS operations of one wave complete in order,
// so the reads need no barrier.
template <int KIND, int TM, int TN, int WM, int WN>
__device__ __forceinline__ void staged_epilogue(const GemmParams& e, int64_t zo, int64_t zi,
                                                int64_t mw, int64_t nw, f32x4 (&acc)[TM][TN],
                                                bf16_t* region) {
  constexpr int U = WN / 8;
  static_assert(WN % 16 == 0 && (WM * U) % 64 == 0, "staged epilogue shape");
  const int lane = threadIdx.x & 63;
  uint8_t* reg = reinterpret_cast<uint8_t*>(region);
  float bias[EpiTraits<KIND>::BIAS ? TN : 1][4];
  load_epi_bias<KIND, TN>(e, nw, bias);
  const bf16_t* rz = EpiTraits<KIND>::RES ? (const bf16_t*)e.res + zo * e.sr_o + zi * e.sr_i : nullptr;
  stage_rows<KIND, TM, TN, WN, 0, TM>(e, rz, mw, nw, acc, bias, reg);
  bf16_t* cz = (bf16_t*)e.C + zo * e.sc_o + zi * e.sc_i;
#pragma unroll
  for (int p = 0; p < WM * U / 64; ++p) {
    const int q = p * 64 + lane, r = q / U, u = q - r * U;
    const uint4 val = *reinterpret_cast<const uint4*>(reg + (r * U + (u + r) % U) * 16);
    const int64_t m = mw + r, n = nw + 8 * u;
    if (m >= e.M || n >= e.N) continue;
    bf16_t* c = cz + m * e.ldc + n;
    if (n + 8 <= e.N) {
      gstore16(c, val);
    } else {  // the row's last piece when N % 8 != 0
      const uint32_t h[4] = {val.x, val.y, val.z, val.w};
#pragma unroll
      for (int t = 0; t < 8; ++t)
        if (n + t < e.N) gstore(c + t, (bf16_t)(h[t >> 1] >> (16 * (t & 1))));
    }
  }
}

// QKV head scatter through LDS (bf16, D a multiple of 8). A wave whose column slab lies in Q
// or K stages its rows as above and writes each 16-byte row piece (8 consecutive d of one
// head) to q[b, h, t, :] or k[b, h, pos0 + t, :]. A slab in V is staged transposed (column c
// holds the WM rows, its 16-byte units rotated by c against bank conflicts) and each unit,
// 8 consecutive rows of one d, goes to vt[b, h, d, pos0 + t .. + 7]: as one 16-byte store
// when T, the cache capacity L and pos0 are multiples of 8 (the 8 rows then share b and the
// destination is aligned), or, with VELEM (any T, L and pos0; ViT-S/4: T = 65), as 8
// 2-byte stores with a (b, t) per row, which still writes runs of consecutive t. Returns
// false (nothing written) for a slab that straddles two parts; the caller then runs the
// generic epilogue for that wave.
template <bool BIAS, int TM, int TN, int WM, int WN, bool VELEM = false>
__device__ __forceinline__ bool staged_qkv_epilogue(const GemmParams& e, int64_t mw, int64_t nw,
                                                    f32x4 (&acc)[TM][TN], bf16_t* region) {
  constexpr int U = WN / 8, RU = WM / 8;
  static_assert(WN % 16 == 0 && (WM * U) % 64 == 0 && WM % 8 == 0, "staged qkv shape");
  const int qw = e.Hq * e.Dh, kw = e.Hkv * e.Dh;
  if (nw >= e.N) return true;  // slab past N: nothing to write
  const int n_lo = (int)nw, n_hi = (int)min(nw + WN, e.N) - 1;
  const int part = n_lo < qw ? 0 : (n_lo < qw + kw ? 1 : 2);
  const int part_hi = n_hi < qw ? 0 : (n_hi < qw + kw ? 1 : 2);
  if (part_hi != part) return false;
  const int lane = threadIdx.x & 63, fr = lane & 15, fc = lane >> 4;
  uint8_t* reg = reinterpret_cast<uint8_t*>(region);
  float bias[BIAS ? TN : 1][4];
  if (BIAS) {
#pragma unroll
    for (int j = 0; j < (BIAS ? TN : 1); ++j) {
      const int64_t n = nw + 16 * j + 4 * fc;
#pragma unroll
      for (int q = 0; q < 4; ++q) bias[j][q] = bias_at(e, n + q);
    }
  }
  const int base = part == 0 ? 0 : (part == 1 ? qw : qw + kw);
  if (part < 2) {
    // destination of this part, selected once: q [B, Hq, T, D] or k [B, Hkv, L, D] at pos0
    const uintptr_t dbase = part == 0 ? (uintptr_t)e.q : (uintptr_t)e.k;
    const int heads = part == 0 ? e.Hq : e.Hkv, tdim = part == 0 ? e.T : e.L;
    const int toff = part == 0 ? 0 : e.pos0;
#pragma unroll
    for (int i = 0; i < TM; ++i) {
      const int r = 16 * i + fr;
#pragma unroll
      for (int j = 0; j < TN; ++j) {
        float v[4] = {acc[i][j][0], acc[i][j][1], acc[i][j][2], acc[i][j][3]};
        if (BIAS) {
#pragma unroll
          for (int q = 0; q < 4; ++q) v[q] = v[q] + bias[BIAS ? j : 0][q];
        }
        uint2 w;
        w.x = (uint32_t)f2bf(v[0]) | ((uint32_t)f2bf(v[1]) << 16);
        w.y = (uint32_t)f2bf(v[2]) | ((uint32_t)f2bf(v[3]) << 16);
        const int u = 2 * j + (fc >> 1);
        *reinterpret_cast<uint2*>(reg + (r * U + (u + r) % U) * 16 + (fc & 1) * 8) = w;
      }
    }
#pragma unroll
    for (int p = 0; p < WM * U / 64; ++p) {
      const int q = p * 64 + lane, r = q / U, u = q - r * U;
      const uint4 val = *reinterpret_cast<const uint4*>(reg + (r * U + (u + r) % U) * 16);
      const int64_t m = mw + r, n = nw + 8 * u;
      if (m >= e.M || n >= e.N) continue;
      const int b = (int)fast_div((uint32_t)m, e.div_T), t = (int)m - b * e.T;
      const int nn = (int)n - base;
      const int h = (int)fast_div((uint32_t)nn, e.div_Dh), d = nn - h * e.Dh;
      gstore16(reinterpret_cast<bf16_t*>(dbase) + ((int64_t)(b * heads + h) * tdim + t + toff) * e.Dh + d, val);
    }
    return true;
  }
  // V: transposed staging, element (column c, row r) at column c's unit (r / 8 + c) % RU
#pragma unroll
  for (int i = 0; i < TM; ++i) {
    const int r = 16 * i + fr;
#pragma unroll
    for (int j = 0; j < TN; ++j) {
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        float v = acc[i][j][q];
        if (BIAS) v = v + bias[BIAS ? j : 0][q];
        const int c = 16 * j + 4 * fc + q;
        *reinterpret_cast<bf16_t*>(reg + (c * RU + ((r >> 3) + c) % RU) * 16 + (r & 7) * 2) = f2bf(v);
      }
    }
  }
#pragma unroll
  for (int p = 0; p < WN * RU / 64; ++p) {
    const int q = p * 64 + lane, c = q / RU, ru = q - c * RU;
    const uint4 val = *reinterpret_cast<const uint4*>(reg + (c * RU + (ru + c) % RU) * 16);
    const int64_t m = mw + 8 * ru, n = nw + c;
    if (m >= e.M || n >= e.N) continue;
    if constexpr (!VELEM) {  // rows m .. m+7 share b and start an aligned run of 8 positions
      const int b = (int)fast_div((uint32_t)m, e.div_T), t = (int)m - b * e.T;
      const int nn = (int)n - base;
      const int h = (int)fast_div((uint32_t)nn, e.div_Dh), d = nn - h * e.Dh;
      gstore16((bf16_t*)e.vt + ((int64_t)(b * e.Hkv + h) * e.Dh + d) * e.L + t + e.pos0, val);
    } else {
      const int nn = (int)n - base;
      const int h = (int)fast_div((uint32_t)nn, e.div_Dh), d = nn - h * e.Dh;
      const uint32_t hw[4] = {val.x, val.y, val.z, val.w};
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const int64_t mj = m + j;
        if (mj >= e.M) break;
        const int b = (int)fast_div((uint32_t)mj, e.div_T), t = (int)mj - b * e.T;
        gstore((bf16_t*)e.vt + ((int64_t)(b * e.Hkv + h) * e.Dh + d) * e.L + t + e.pos0,
               (bf16_t)(hw[j >> 1] >> (16 * (j & 1))));
      }
    }
  }
  return true;
}

// Gated (GeGLU) epilogue through LDS: columns come in (gate f, up f) pairs, so a lane's 4
// results give 2 outputs act(gate) * up; the wave's WN / 2 output columns are staged as
// packed pairs and written as 16-byte row pieces (bf16, no bias, N / 2 % 8 == 0).
template <int KIND, int TM, int TN, int WM, int WN>
__device__ __forceinline__ void staged_geglu_epilogue(const GemmParams& e, int64_t zo, int64_t zi,
                                                      int64_t mw, int64_t nw,
                                                      f32x4 (&acc)[TM][TN], bf16_t* region) {
  constexpr int U = WN / 16;  // 16-byte output pieces per row (8 outputs each)
  static_assert(WN % 16 == 0 && (WM * U) % 64 == 0, "staged gated shape");
  const int lane = threadIdx.x & 63, fr = lane & 15, fc = lane >> 4;
  uint8_t* reg = reinterpret_cast<uint8_t*>(region);
#pragma unroll
  for (int i = 0; i < TM; ++i) {
    const int r = 16 * i + fr;
#pragma unroll
    for (int j = 0; j < TN; ++j) {
      const f32x4 v = acc[i][j];
      const float h0 = (KIND == EPI_GEGLU_GELU ? gelu_tanh(v[0]) : silu_tanh(v[0])) * v[1];
      const float h1 = (KIND == EPI_GEGLU_GELU ? gelu_tanh(v[2]) : silu_tanh(v[2])) * v[3];
      // output columns 8 j + 2 fc, +1 of this wave: piece j, bytes 4 fc
      *reinterpret_cast<uint32_t*>(reg + (r * U + (j + r) % U) * 16 + 4 * fc) =
          (uint32_t)f2bf(h0) | ((uint32_t)f2bf(h1) << 16);
    }
  }
  bf16_t* cz = (bf16_t*)e.C + zo * e.sc_o + zi * e.sc_i;
  const int64_t nout = e.N / 2, ow = nw / 2;
#pragma unroll
  for (int p = 0; p < WM * U / 64; ++p) {
    const int q = p * 64 + lane, r = q / U, u = q - r * U;
    const uint4 val = *reinterpret_cast<const uint4*>(reg + (r * U + (u + r) % U) * 16);
    const int64_t m = mw + r, n = ow + 8 * u;
    if (m >= e.M || n >= nout) continue;
    gstore16(cz + m * e.ldc + n, val);
  }
}

}  // namespace tl
