// Internal structures shared by the gemm kernels (gemm.hip, gemm_fp8.hip).
#pragma once

#include <type_traits>

#include "common.h"

namespace th {

struct EpiOutK {
  int op, a, b, e;
  void* ptr;
  int64_t ld;
  int dtype, vec;  // vec: 4-element vector access possible
  int vec8;        // 8-element (16-byte bf16 / 2 x 16-byte fp32) access possible
  int cb, ce;      // accumulator columns [cb, ce) land at output columns 0 .. ce - cb
};

struct GemmK {
  const void* A;
  int64_t lda;
  const void* B;
  int64_t ldb;
  int64_t M, N, K;
  int tiles_m, tiles_n;
  int bn, n_acc;
  int sumsq;
  unsigned rscale_mask;
  float inv_k, eps;
  const void* extra[TH_MAX_EXTRA];
  int64_t ld_extra[TH_MAX_EXTRA];
  int extra_dtype[TH_MAX_EXTRA];
  int extra_vec[TH_MAX_EXTRA];
  int extra_vec8[TH_MAX_EXTRA];
  const float* rcos;
  const float* rsin;
  int hd, period;
  int n_out;
  int asplit;  // persistent kernel: each wave's column half is one whole accumulator (n_acc == 2)
  int pair_hd; // ping-pong kernel: head dim (64 or wider) whose halves are paired in a wave, else 0
  EpiOutK out[TH_MAX_OUT];
  float* sumsq_out;
  const float* gain;  // optional [K]: products use lhs[m, k] * gain[k] (fp8 path); sumsq stays unscaled
  // optional [M][n_rs_parts] (row stride ld_rs_parts): each row's sum of squares as
  // partial sums made by the lhs's producer, summed in order instead of sum_k lhs^2
  const float* rs_parts;
  int64_t ld_rs_parts;
  int n_rs_parts;
  // optional (fp8 path): output gain_index stored as bf16(bf16(v) * gain_out[n]),
  // each row's sums of bf16(v)^2 per 256 columns to ss_parts_out
  const float* gain_out;
  float* ss_parts_out;
  int64_t ld_ss_parts_out;
  int gain_index;
};

// Row `row`'s sum of squares: `own` (the kernel's sum over its lhs fragments), or
// the sum of the producer's partial sums when the caller gave them, added one
// after another in order; rows past M read row M - 1, whose scale is never
// used. The parts are fetched 32 at a time, every load issued before the
// first addition (indices clamped, additions past the end selected away: no
// branch for the compiler to put a wait into), so a row costs one memory
// round trip per 32 parts instead of one per 4.
__device__ __forceinline__ float row_parts_sum(const float4* q, int n4) {
  float v = 0.f;
  for (int i0 = 0; i0 < n4; i0 += 8) {
    float4 f[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) f[j] = q[i0 + j < n4 ? i0 + j : n4 - 1];
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      float t = v + f[j].x;
      t += f[j].y;
      t += f[j].z;
      t += f[j].w;
      v = i0 + j < n4 ? t : v;
    }
  }
  return v;
}

__device__ __forceinline__ float row_sumsq(const GemmK& p, int64_t row, float own) {
  if (p.rs_parts == nullptr) return own;
  return row_parts_sum((const float4*)(p.rs_parts + (row < p.M ? row : p.M - 1) * p.ld_rs_parts), p.n_rs_parts >> 2);
}

// fp8-weight path (gemm_fp8.hip)
struct Fp8K {
  GemmK k;           // output ops, row scale, extras, RoPE tables
  const void* A;     // bf16 [M, K]
  int64_t lda;
  const void* B;     // packed e4m3 rhs, K contiguous
  int64_t ldb;       // bytes per packed row
  int64_t M, N, K, Npk, bn;
  const float* scale;  // [n_acc][N]
  int splits;
  int64_t ksplit;
  float* part;       // [splits][M][Npk]
  float* sumsq_part; // [splits][M]
  int fused;         // one split finishing its tiles in the main kernel (no reduce pass)
  int ss_pre;        // row sums of squares already in sumsq_part (split 0; the others zero)
};

// 4 consecutive elements (one 8-byte bf16 / 16-byte fp32 access when vec,
// element by element for a ragged end or unaligned rows).
__device__ __forceinline__ float4 load4(const void* p, int64_t off, int dtype, bool vec, int valid) {
  float4 v = make_float4(0.f, 0.f, 0.f, 0.f);
  if (vec && valid >= 4) {
    if (dtype == TH_BF16) {
      const uint2 w = *(const uint2*)((const uint16_t*)p + off);
      v.x = __uint_as_float(w.x << 16);
      v.y = __uint_as_float(w.x & 0xffff0000u);
      v.z = __uint_as_float(w.y << 16);
      v.w = __uint_as_float(w.y & 0xffff0000u);
    } else {
      v = *(const float4*)((const float*)p + off);
    }
    return v;
  }
  float t[4] = {0.f, 0.f, 0.f, 0.f};
  for (int q = 0; q < 4 && q < valid; ++q) t[q] = load_elem(p, off + q, dtype);
  return make_float4(t[0], t[1], t[2], t[3]);
}

__device__ __forceinline__ void store4(void* p, int64_t off, int dtype, bool vec, int valid, float4 v) {
  if (vec && valid >= 4) {
    if (dtype == TH_BF16) {
      uint2 w;
      w.x = pk_bf16x2(v.x, v.y);
      w.y = pk_bf16x2(v.z, v.w);
      *(uint2*)((uint16_t*)p + off) = w;
    } else {
      *(float4*)((float*)p + off) = v;
    }
    return;
  }
  const float t[4] = {v.x, v.y, v.z, v.w};
  for (int q = 0; q < 4 && q < valid; ++q) store_elem(p, off + q, dtype, t[q]);
}

// 8 consecutive elements (one 16-byte bf16 or two 16-byte fp32 accesses when
// vec8, element by element for a ragged end or unaligned rows).
__device__ __forceinline__ void store8(void* p, int64_t off, int dtype, bool vec8, int valid, const float* v) {
  if (vec8 && valid >= 8) {
    if (dtype == TH_BF16) {
      uint4 w;
      w.x = pk_bf16x2(v[0], v[1]);
      w.y = pk_bf16x2(v[2], v[3]);
      w.z = pk_bf16x2(v[4], v[5]);
      w.w = pk_bf16x2(v[6], v[7]);
      *(uint4*)((uint16_t*)p + off) = w;
    } else {
      *(float4*)((float*)p + off) = make_float4(v[0], v[1], v[2], v[3]);
      *(float4*)((float*)p + off + 4) = make_float4(v[4], v[5], v[6], v[7]);
    }
    return;
  }
#pragma unroll
  for (int q = 0; q < 8; ++q)
    if (q < valid) store_elem(p, off + q, dtype, v[q]);
}

// Outputs o and o + 1 compute the same values (same op, operands and column
// window; only the destination differs).
__host__ __device__ __forceinline__ bool same_values(const EpiOutK& x, const EpiOutK& y) {
  return x.op == y.op && x.a == y.a && x.b == y.b && x.e == y.e && x.cb == y.cb && x.ce == y.ce;
}

// What a GEMM's epilogue adds to the time of a tile, in the terms of the estimates that
// choose a main loop. An output that repeats the one before it (an fp32 copy) counts for
// nothing, so that a value's bits do not depend on whether a copy is stored beside it.
struct EpiCost {
  double rope;  // share of the columns that are rotated
  double wide;  // bytes stored and loaded per column beyond the 4 that every loop hides
  bool ragged;  // output rows that are not whole 128-byte lines
  bool extra;   // an operand per element
  int outs;
};

inline EpiCost gemm_epi_cost(const GemmK& k) {
  EpiCost c{0, 0, false, false, 0};
  double bytes = 0;
  const double cols = (double)k.N * k.n_acc;
  for (int o = 0; o < k.n_out; ++o) {
    const EpiOutK& eo = k.out[o];
    if (o > 0 && same_values(k.out[o - 1], eo)) continue;
    const double w = (double)(eo.ce - eo.cb) / cols;
    bytes += 2 * w;
    if (eo.e >= 0) bytes += w * (k.extra_dtype[eo.e] == TH_F32 ? 4 : 2);
    if (eo.op == TH_EPI_ROPE || eo.op == TH_EPI_ROPE_PAIR) c.rope += w;
    c.ragged |= eo.ld % 64 != 0 && eo.op != TH_EPI_SWIGLU;  // (SwiGLU is stored from registers in every loop)
    c.extra |= eo.e >= 0;
    ++c.outs;
  }
  c.wide = bytes > 4 ? bytes - 4 : 0;
  return c;
}

// ping-pong persistent bf16 kernel (gemm_pp.hip)
bool gemm_pp_fits(const GemmK& k);
int gemm_pp_rows(const GemmK& k, const EpiCost& ec, int64_t cus, double* us);
int launch_gemm_pp(const GemmK& k, int bm, hipStream_t s);

int64_t fp8_workspace_bytes(int64_t M, int64_t Npk, int64_t K, int bn, int n_acc);
int launch_gemm_fp8(const GemmK& k, int64_t Npk, const float* scale, float* ws, int64_t ws_bytes, hipStream_t s);

}  // namespace th
