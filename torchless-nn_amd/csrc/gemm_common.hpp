// Shared pieces of the GEMM kernels (gemm.hip, gemm_rows.hip, gemm_split.hip): the parameter
// block, global-memory access helpers, the general epilogue and the output tile order.
#pragma once

#include "tl_internal.hpp"

namespace tl {

// Epilogues of the LDS-staged path, one compiled variant each (bias, activation and
// residual known at compile time, so the fragment loops carry no per-element tests);
// EPI_GENERIC keeps mfma_epilogue (QKV scatter, GeGLU, fp32 output, divisor, unaligned
// residual rows or output rows).
enum EpiKind { EPI_GENERIC = 0, EPI_PLAIN, EPI_BIAS, EPI_BIAS_GELU, EPI_BIAS_SILU, EPI_BIAS_RES, EPI_RES,
               EPI_QKV, EPI_QKV_BIAS, EPI_GEGLU_GELU, EPI_GEGLU_SILU };

struct GemmParams {
  const void* A;
  const void* B;
  void* C;
  int64_t M, N, K, lda, ldb, ldc;
  int64_t batch_inner;
  int64_t sa_o, sa_i, sb_o, sb_i, sc_o, sc_i;
  const void* bias;
  const void* res;
  int64_t ldr, sr_o, sr_i;
  float divisor;
  int act;
  int b_kn;
  int vec_store;
  int vec_res;  // residual rows allow one 4-element vector load per lane fragment
  int epi;      // EpiKind: which specialised LDS-staged epilogue applies (bf16 output)
  int qkv;
  void* q;
  void* k;
  void* vt;
  int T, Hq, Hkv, Dh;
  int L, pos0;  // key/value cache capacity and write position (QKV split)
  const int64_t* pos0_dev;  // when set: the write position, read from device memory
  int geglu;    // gated epilogue: C[m, n/2] = act(acc[m, n]) * acc[m, n+1]
  int tiles_m, tiles_n, group_m;
  FastDiv div_T, div_Dh;
  // RMS row scaling (skinny kernel): the product of row m is multiplied by
  // 1 / sqrt(sum_k A[m, k]^2 / K + norm_eps) before the epilogue, which with the norm's gain
  // folded into B makes it RMSNorm(A) @ B
  int norm_rows;
  float norm_eps;
};

// Global-memory access through an address-space-1 pointer. The epilogue's pointers come
// from the parameter block, so the compiler cannot prove they are global and would emit
// flat instructions, which also count in the LDS wait counter: every wait for an LDS read
// would then wait for the stores issued before it as well.
// (HIP's uint2/uint4 are C++ structs whose assignment takes a generic `this`, so 8- and
// 16-byte accesses go through native vector types.)
template <typename T>
__device__ __forceinline__ void gstore(T* p, const T& v) {
  *(__attribute__((address_space(1))) T*)p = v;
}
template <typename T>
__device__ __forceinline__ T gload(const T* p) {
  return *(const __attribute__((address_space(1))) T*)p;
}
typedef uint32_t u32x2_t __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));
__device__ __forceinline__ void gstore16(void* p, uint4 v) {
  const u32x4_t t = {v.x, v.y, v.z, v.w};
  *(__attribute__((address_space(1))) u32x4_t*)p = t;
}
__device__ __forceinline__ void gstore8(void* p, uint2 v) {
  const u32x2_t t = {v.x, v.y};
  *(__attribute__((address_space(1))) u32x2_t*)p = t;
}
__device__ __forceinline__ uint2 gload8(const void* p) {
  const u32x2_t t = *(const __attribute__((address_space(1))) u32x2_t*)p;
  return make_uint2(t.x, t.y);
}
template <typename T>
__device__ __forceinline__ void gstore_elem(T* p, float v) {
  if (sizeof(T) == 4) gstore(reinterpret_cast<float*>(p), v);
  else gstore(reinterpret_cast<bf16_t*>(p), f2bf(v));
}
template <typename T>
__device__ __forceinline__ float gload_elem(const T* p) {
  if (sizeof(T) == 4) return gload(reinterpret_cast<const float*>(p));
  return bf2f(gload(reinterpret_cast<const bf16_t*>(p)));
}
__device__ __forceinline__ void gstore_f4(float* p, const float (&v)[4]) {
  gstore16(p, make_uint4(__float_as_uint(v[0]), __float_as_uint(v[1]), __float_as_uint(v[2]),
                         __float_as_uint(v[3])));
}
__device__ __forceinline__ void gload_f4(const float* p, float (&v)[4]) {
  const u32x4_t t = *(const __attribute__((address_space(1))) u32x4_t*)p;
  v[0] = __uint_as_float(t.x); v[1] = __uint_as_float(t.y);
  v[2] = __uint_as_float(t.z); v[3] = __uint_as_float(t.w);
}

// Bias value of column n, 0 past N. The load itself is unconditional (column clamped to
// N - 1) and the value is selected afterwards: a load under a per-lane condition compiles to
// its own exec-masked branch that waits for it, so a fragment's loads would complete one
// after another instead of together.
template <typename TI = bf16_t>
__device__ __forceinline__ float bias_at(const GemmParams& e, int64_t n) {
  const float b = gload_elem((const TI*)e.bias + (n < e.N ? n : e.N - 1));
  return n < e.N ? b : 0.f;
}

// Applies the epilogue to 4 consecutive columns n0..n0+3 of row m and stores them.
template <typename TI, typename TO>
__device__ __forceinline__ void epilogue4(const GemmParams& p, int64_t zo, int64_t zi, int64_t m,
                                          int64_t n0, float v[4]) {
  if (m >= p.M || n0 >= p.N) return;
  const int cnt = p.N - n0 >= 4 ? 4 : (int)(p.N - n0);
  if (p.divisor != 1.0f) {
#pragma unroll
    for (int e = 0; e < 4; ++e) v[e] = v[e] / p.divisor;
  }
  if (p.bias) {  // unconditional loads (clamped to column N - 1), selected afterwards
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const float b = gload_elem((const TI*)p.bias + (e < cnt ? n0 + e : p.N - 1));
      if (e < cnt) v[e] = v[e] + b;
    }
  }
  if (p.geglu) {  // columns (gate f, up f, gate f+1, up f+1), n0 even
    TO* c = (TO*)p.C + zo * p.sc_o + zi * p.sc_i + m * p.ldc + n0 / 2;
    gstore_elem(c, apply_act(v[0], p.act) * v[1]);
    if (cnt == 4) gstore_elem(c + 1, apply_act(v[2], p.act) * v[3]);
    return;
  }
  if (p.act != TL_ACT_NONE) {
#pragma unroll
    for (int e = 0; e < 4; ++e) v[e] = apply_act(v[e], p.act);
  }
  if (p.res) {
    const TO* r = (const TO*)p.res + zo * p.sr_o + zi * p.sr_i + m * p.ldr;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const float x = gload_elem(r + (e < cnt ? n0 + e : p.N - 1));
      if (e < cnt) v[e] = v[e] + x;
    }
  }
  if (p.qkv) {
    // Dh % 4 == 0 (checked on the host), so the 4 columns share one head of one part.
    const int mi = (int)m, ni = (int)n0;
    const int b = mi / p.T, t = mi - b * p.T;
    const int pos0 = p.pos0_dev ? (int)*p.pos0_dev : p.pos0;
    const int qw = p.Hq * p.Dh, kw = p.Hkv * p.Dh;
    TO* dst;
    int64_t step;
    if (ni < qw) {
      const int h = ni / p.Dh, d = ni - h * p.Dh;
      dst = (TO*)p.q + ((int64_t)(b * p.Hq + h) * p.T + t) * p.Dh + d;
      step = 1;
    } else if (ni < qw + kw) {
      if (t + pos0 >= p.L) return;  // a device position past the cache: nothing written
      const int nn = ni - qw, h = nn / p.Dh, d = nn - h * p.Dh;
      dst = (TO*)p.k + ((int64_t)(b * p.Hkv + h) * p.L + t + pos0) * p.Dh + d;
      step = 1;
    } else {
      if (t + pos0 >= p.L) return;
      const int nn = ni - qw - kw, h = nn / p.Dh, d = nn - h * p.Dh;
      dst = (TO*)p.vt + ((int64_t)(b * p.Hkv + h) * p.Dh + d) * p.L + t + pos0;
      step = p.L;
    }
    if (step == 1 && sizeof(TO) == 2) {
      uint2 w;
      w.x = (uint32_t)f2bf(v[0]) | ((uint32_t)f2bf(v[1]) << 16);
      w.y = (uint32_t)f2bf(v[2]) | ((uint32_t)f2bf(v[3]) << 16);
      gstore8(dst, w);
    } else {
#pragma unroll
      for (int e = 0; e < 4; ++e) gstore_elem(dst + e * step, v[e]);
    }
    return;
  }
  TO* c = (TO*)p.C + zo * p.sc_o + zi * p.sc_i + m * p.ldc + n0;
  if (cnt == 4 && p.vec_store) {
    if (sizeof(TO) == 4) {
      gstore_f4(reinterpret_cast<float*>(c), *reinterpret_cast<const float(*)[4]>(v));
    } else {
      uint2 w;
      w.x = (uint32_t)f2bf(v[0]) | ((uint32_t)f2bf(v[1]) << 16);
      w.y = (uint32_t)f2bf(v[2]) | ((uint32_t)f2bf(v[3]) << 16);
      gstore8(c, w);
    }
  } else {
    for (int e = 0; e < cnt; ++e) gstore_elem(c + e, v[e]);
  }
}

// For kernels whose first argument is a GemmParams by value, at offset 0 of the kernarg segment.
// The epilogue re-reads it through an opaque copy of the segment pointer: those loads
// cannot be hoisted to the kernel entry, so the ~40 scalar registers of epilogue fields
// are not held across the K loop (holding them made the large tiles spill to scratch).
typedef __attribute__((address_space(4))) const uint32_t ConstU32;
__device__ __forceinline__ GemmParams late_params() {
  static_assert(sizeof(GemmParams) % 4 == 0, "GemmParams must be whole dwords");
  ConstU32* src = (ConstU32*)__builtin_amdgcn_kernarg_segment_ptr();
  asm volatile("" : "+s"(src));
  GemmParams e;
  uint32_t* dst = reinterpret_cast<uint32_t*>(&e);
#pragma unroll
  for (int i = 0; i < (int)(sizeof(GemmParams) / 4); ++i) dst[i] = src[i];
  return e;
}

// Epilogue of an MFMA accumulator block: acc[i][j] holds rows mb + 16 i and columns
// nb + 16 j .. +3 of this lane. Bias is loaded once per column fragment, 64-bit row
// addresses once per row, and the head scatter splits rows (batch, time) and columns
// (part, head, d) with one fast division each.
template <typename TO, int TM, int TN, typename TI = bf16_t>
__device__ __forceinline__ void mfma_epilogue(const GemmParams& e, int64_t zo, int64_t zi,
                                              int64_t mb, int64_t nb, f32x4 (&acc)[TM][TN]) {
  int cnt[TN];
  float bias[TN][4];
#pragma unroll
  for (int j = 0; j < TN; ++j) {
    const int64_t n = nb + 16 * j;
    cnt[j] = n >= e.N ? 0 : (e.N - n >= 4 ? 4 : (int)(e.N - n));
  }
  // one branch around all the bias loads (a branch per load would wait inside each)
  if (e.bias) {
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int q = 0; q < 4; ++q) bias[j][q] = bias_at<TI>(e, nb + 16 * j + q);
  } else {
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int q = 0; q < 4; ++q) bias[j][q] = 0.f;
  }
  auto finish = [&](float (&v)[4], int j) {
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      if (e.divisor != 1.0f) v[q] = v[q] / e.divisor;
      v[q] = v[q] + bias[j][q];
      if (e.act != TL_ACT_NONE && !e.geglu) v[q] = apply_act(v[q], e.act);
    }
  };
  if (e.qkv) {
    // column split, once per fragment: part (Q, K or V), head h, offset d
    const int qw = e.Hq * e.Dh, kw = e.Hkv * e.Dh;
    TO* cbase[TN];
    int part[TN];
#pragma unroll
    for (int j = 0; j < TN; ++j) {
      const int n = (int)(nb + 16 * j);
      part[j] = n < qw ? 0 : (n < qw + kw ? 1 : 2);
      const int nn = n - (part[j] == 0 ? 0 : (part[j] == 1 ? qw : qw + kw));
      const int h = (int)fast_div((uint32_t)nn, e.div_Dh), d = nn - h * e.Dh;
      cbase[j] = part[j] == 0 ? (TO*)e.q + ((int64_t)h * e.T) * e.Dh + d
               : part[j] == 1 ? (TO*)e.k + ((int64_t)h * e.L) * e.Dh + d
                              : (TO*)e.vt + ((int64_t)h * e.Dh + d) * e.L;
    }
#pragma unroll
    for (int i = 0; i < TM; ++i) {
      const int64_t m = mb + 16 * i;
      if (m >= e.M) continue;
      const int b = (int)fast_div((uint32_t)m, e.div_T), t = (int)m - b * e.T;
      const int pos0 = e.pos0_dev ? (int)*e.pos0_dev : e.pos0;
      const bool in_cache = t + pos0 < e.L;  // a device position past the cache: no K/V rows
      const int64_t rq = ((int64_t)b * e.Hq * e.T + t) * e.Dh;
      const int64_t rk = ((int64_t)b * e.Hkv * e.L + t + pos0) * e.Dh;
      const int64_t rv = (int64_t)b * e.Hkv * e.Dh * e.L + t + pos0;
#pragma unroll
      for (int j = 0; j < TN; ++j) {
        if (cnt[j] == 0) continue;
        float v[4] = {acc[i][j][0], acc[i][j][1], acc[i][j][2], acc[i][j][3]};
        finish(v, j);
        if (part[j] > 0 && !in_cache) continue;
        if (part[j] < 2) {
          TO* dst = cbase[j] + (part[j] == 0 ? rq : rk);
          if (sizeof(TO) == 2) {
            uint2 w;
            w.x = (uint32_t)f2bf(v[0]) | ((uint32_t)f2bf(v[1]) << 16);
            w.y = (uint32_t)f2bf(v[2]) | ((uint32_t)f2bf(v[3]) << 16);
            gstore8(dst, w);
          } else {
#pragma unroll
            for (int q = 0; q < 4; ++q) gstore_elem(dst + q, v[q]);
          }
        } else {
          TO* dst = cbase[j] + rv;
#pragma unroll
          for (int q = 0; q < 4; ++q) gstore_elem(dst + (int64_t)q * e.L, v[q]);
        }
      }
    }
    return;
  }
  TO* cz = (TO*)e.C + zo * e.sc_o + zi * e.sc_i;
  if (e.geglu) {  // columns (gate f, up f, gate f+1, up f+1) with f = n / 2
#pragma unroll
    for (int i = 0; i < TM; ++i) {
      const int64_t m = mb + 16 * i;
      if (m >= e.M) continue;
      TO* crow = cz + m * e.ldc + nb / 2;
#pragma unroll
      for (int j = 0; j < TN; ++j) {
        if (cnt[j] == 0) continue;
        float v[4] = {acc[i][j][0], acc[i][j][1], acc[i][j][2], acc[i][j][3]};
        finish(v, j);
        const float h0 = apply_act(v[0], e.act) * v[1], h1 = apply_act(v[2], e.act) * v[3];
        TO* c = crow + 8 * j;
        if (sizeof(TO) == 2 && cnt[j] == 4 && e.vec_store) {
          gstore(reinterpret_cast<uint32_t*>(c), (uint32_t)f2bf(h0) | ((uint32_t)f2bf(h1) << 16));
        } else {
          gstore_elem(c, h0);
          if (cnt[j] == 4) gstore_elem(c + 1, h1);
        }
      }
    }
    return;
  }
  const TO* rz = e.res ? (const TO*)e.res + zo * e.sr_o + zi * e.sr_i : nullptr;
#pragma unroll
  for (int i = 0; i < TM; ++i) {
    const int64_t m = mb + 16 * i;
    // the row's vector residual pieces, requested together before any is used (reads of
    // rows past M or of fragments that end past N are clamped in bounds and not used)
    float rq[TN][4];
    if (rz && e.vec_res) {
      const TO* r0 = rz + (m < e.M ? m : e.M - 1) * e.ldr;
#pragma unroll
      for (int j = 0; j < TN; ++j) {
        const int64_t c = nb + 16 * j;
        const TO* src = r0 + (c + 4 <= e.N ? c : 0);
        if constexpr (sizeof(TO) == 2) {
          const uint2 u = gload8(src);
          rq[j][0] = __uint_as_float(u.x << 16); rq[j][1] = __uint_as_float(u.x & 0xffff0000u);
          rq[j][2] = __uint_as_float(u.y << 16); rq[j][3] = __uint_as_float(u.y & 0xffff0000u);
        } else {
          gload_f4(reinterpret_cast<const float*>(src), rq[j]);
        }
      }
    }
    if (m >= e.M) continue;
    TO* crow = cz + m * e.ldc + nb;
    const TO* rrow = rz ? rz + m * e.ldr + nb : nullptr;
#pragma unroll
    for (int j = 0; j < TN; ++j) {
      if (cnt[j] == 0) continue;
      float v[4] = {acc[i][j][0], acc[i][j][1], acc[i][j][2], acc[i][j][3]};
      finish(v, j);
      if (rrow) {
        if (cnt[j] == 4 && e.vec_res) {
#pragma unroll
          for (int q = 0; q < 4; ++q) v[q] = v[q] + rq[j][q];
        } else {
#pragma unroll
          for (int q = 0; q < 4; ++q)
            if (q < cnt[j]) v[q] = v[q] + gload_elem(rrow + 16 * j + q);
        }
      }
      TO* c = crow + 16 * j;
      if (cnt[j] == 4 && e.vec_store) {
        if (sizeof(TO) == 4) {
          gstore_f4(reinterpret_cast<float*>(c), v);
        } else {
          uint2 w;
          w.x = (uint32_t)f2bf(v[0]) | ((uint32_t)f2bf(v[1]) << 16);
          w.y = (uint32_t)f2bf(v[2]) | ((uint32_t)f2bf(v[3]) << 16);
          gstore8(c, w);
        }
      } else {
        for (int q = 0; q < cnt[j]; ++q) gstore_elem(c + q, v[q]);
      }
    }
  }
}

// Position i of the grouped tile order -> output tile (tm, tn): groups of group_m
// tile-rows, walked row-fastest.
__device__ __forceinline__ void grouped_tile(int i, const GemmParams& p, int& tm, int& tn) {
  const int per_group = p.group_m * p.tiles_n;
  const int g = i / per_group;
  const int first_m = g * p.group_m;
  const int gm = min(p.tiles_m - first_m, p.group_m);
  const int k = i - g * per_group;
  tm = first_m + k % gm;
  tn = k / gm;
}

// Block id -> output tile: workgroups are dispatched round-robin over the 8 XCDs, so XCD x
// runs blocks x, x+8, ...; give it the contiguous run [x q + min(x, r), ...) of the
// grouped order.
__device__ __forceinline__ void map_tile(int bid, const GemmParams& p, int& tm, int& tn) {
  const int ntiles = p.tiles_m * p.tiles_n;
  const int x = bid & 7, local = bid >> 3;
  const int q = ntiles >> 3, r = ntiles & 7;
  grouped_tile(x * q + min(x, r) + local, p, tm, tn);
}

// Scheduling pattern for one K step of fragment reads and MFMAs: NR reads of the first
// half, then the second half's NR reads each followed by a share of the first half's NM
// MFMAs, then the second half's NM MFMAs. The fragment registers of both halves stay live,
// so no MFMA waits for an LDS read issued right before it.
template <int NR, int NM, int R = 0>
__device__ __forceinline__ void interleave_reads_mfma() {
  if constexpr (R < NR) {
    constexpr int q = NM / NR, rem = NM % NR;
    __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);                       // DS read
    __builtin_amdgcn_sched_group_barrier(0x008, q + (R < rem ? 1 : 0), 0);  // MFMA
    interleave_reads_mfma<NR, NM, R + 1>();
  }
}
template <int NR, int NM>
__device__ __forceinline__ void schedule_kstep() {
  __builtin_amdgcn_sched_group_barrier(0x100, NR, 0);
  interleave_reads_mfma<NR, NM>();
  __builtin_amdgcn_sched_group_barrier(0x008, NM, 0);
}

}  // namespace tl
