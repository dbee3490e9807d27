// The bf16 GEMM's large-tile main loop: persistent workgroups of eight waves on
// (64 TM) x 256 output tiles, TM = 2, 3 or 4, with the two waves of a SIMD
// offset by half a phase (one reads LDS and issues loads while the other's
// MFMAs run).
//
// What bounds it: MFMA issue. A 256 x 256 x 64 step is 2048 cycles of
// v_mfma_f32_32x32x16_bf16 per SIMD; the loop has to keep 64 KB of operand
// loads per step in flight (L2 and HBM latency is about one step), read
// 192 KB of fragments out of LDS, and lose nothing at its barriers.
//
// * Waves: wm = wave / 4 owns half the rows, wn = wave % 4 owns two 32-column
//   subtiles. Waves w and w + 4 share a SIMD, so the two row halves are the two
//   groups of the half-phase offset: the second group passes one extra barrier
//   at the start of a tile, the first one at its end.
// * A K step (64 deep) is four phases; each multiplies one half of the wave's
//   row subtiles (A0, A1) by one of its column subtiles (B0, B1):
//     phase 0  A0 B0   reads A0(kt)     loads B0(kt + 2)
//     phase 1  A0 B1   reads B1(kt)     loads A0(kt + 2)
//     phase 2  A1 B1   reads A1(kt)     loads B1(kt + 2)
//     phase 3  A1 B0   reads B0(kt + 1) loads A1(kt + 2)
//   A phase is: read fragments, issue loads, wait for the region the next phase
//   reads (loads issued six phases ago) and for the own reads, barrier, MFMAs,
//   barrier. Every region of the two LDS stages is refilled one phase after its
//   last read, so a load has six phases (one and a half K steps) to land where
//   a whole-stage double buffer gives it less than one.
//   The next B0 lands in B1's registers: the two swap roles every K step.
//   That holds only while the compiler adds no wait of its own to the loop: a load
//   of the epilogue that may still be pending on some path, or a spilled register
//   reloaded, makes it wait for every load in flight (tests/test_gemm_pp_schedule.py
//   reads the assembly). So the epilogue loads nothing that it does not use, and with
//   256 rows the per-lane offsets are computed anew for each K loop instead of kept
//   across the epilogue. (With such waits in 192-row tiles and spills in 256-row ones: fused RoPE
//   16384 x 4096 x 4096 524 us, without 449; 16384 x 50280 x 1024 1756, without 1612;
//   SwiGLU 3001 x 2 * 14336 x 4096 591, without 566.)
// * K need only be a multiple of 8: the last two steps re-read columns, whose
//   fragments are zeroed. (Two steps, so that the step count is even and every
//   tile starts in stage 0 with B0 in the same registers; a branch on the
//   parity around the last steps made the compiler copy the accumulators.)
// * Column subtiles of a fused RoPE output are paired: subtile 1 holds the
//   rotation partners of subtile 0 (half a head away), so a head as wide as the
//   tile never needs another wave.
// * The products are formed transposed (weights as the MFMA's first operand), so
//   a lane holds one output row and runs of four consecutive columns. A
//   v_permlane32_swap per pair of values makes them runs of eight, and a
//   v_permlane16_swap puts the four runs of a subtile's row into four lanes of
//   one register: the epilogue works on registers alone, without LDS or
//   barriers, its accesses 16 bytes per lane and 64 consecutive bytes per row
//   (32 bytes per row, without the second swap, made a SwiGLU tile's stores 14%
//   of a K = 1024 launch slower), and the next tile's first two K steps load
//   under it.
#include <algorithm>

#include "gemm_internal.h"

namespace th {

namespace {

// Output tile of persistent step L: XCD x (workgroups x, x + 8, ...) walks one
// contiguous range of tiles, 8 tile rows at a time, for any number of tiles.
__device__ __forceinline__ void pp_map(int L, int tiles_m, int tiles_n, int& tm, int& tn) {
  const int nb = tiles_m * tiles_n, q = nb >> 3, r = nb & 7, x = L & 7;
  const int pid = x * q + min(x, r) + (L >> 3);
  const int G = 8, group = pid / (G * tiles_n), first = group * G;
  const int gm = min(tiles_m - first, G), in_group = pid - group * G * tiles_n;
  tm = first + in_group % gm;
  tn = in_group / gm;
}

// The lane id, computed anew where it is asked for: what is derived from it there
// is not kept in registers across a loop that has none to spare.
__device__ __forceinline__ int fresh_lane() {
  int l;
  asm volatile("v_mbcnt_lo_u32_b32 %0, -1, 0\n\tv_mbcnt_hi_u32_b32 %0, -1, %0" : "=v"(l));
  return l;
}

// The kernel's arguments, read anew where they are asked for: values derived from
// them (and from the lane id, fresh_lane) per tile would otherwise be kept in
// registers across the K loop, which has none to spare (spilled, their reload in
// the epilogue waits for the next tile's loads, which are issued before it).
__device__ __forceinline__ const GemmK& fresh_args() {
  auto a = (const __attribute__((address_space(4))) GemmK*)__builtin_amdgcn_kernarg_segment_ptr();
  asm volatile("" : "+s"(a));
  return *(const GemmK*)a;
}

typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));

// Buffer access to one wave's rows of an output or operand: the base is uniform, a lane's
// offset 32 bits, and a lane with nothing to access has the offset kNone (or kNone and less than
// 2 GiB more), which is past the end: its load is zero and its store dropped without a branch. (The compiler counts what is
// in flight through straight-line code; around a branch it waits for everything.)
constexpr uint32_t kNone = 0x80000000u;
__device__ __forceinline__ auto wave_rows(const void* p, int64_t byte_off) {
  return __builtin_amdgcn_make_buffer_rsrc((void*)((char*)p + byte_off), 0, 0x7fffffff, 0x00020000);
}

// acc[T] of this wave, lanes traded: afterwards octet s[u][q] of lane l is row 16 q + l % 16,
// columns 8 (l / 32 + 2 (l / 16 % 2)) .. + 8 of column subtile u (NU of them).
// Before, registers 8 q + j hold row l % 32, columns 16 q + 4 (l / 32) + j, and registers
// 8 q + 4 + j the columns 8 further on. Swapping the upper half of registers 8 q + j with the
// lower half of 8 q + 4 + j leaves columns 16 q + 8 (l / 32) + j and + 4 + j. Then q = 0 and 1
// trade their odd and even rows of 16 lanes: q becomes the row half, and lane bits 5 and 4 are
// column bits 3 and 4.
template <int NU>
__device__ __forceinline__ void trade_lanes(float (&s)[2][2][8]) {
#pragma unroll
  for (int u = 0; u < NU; ++u) {
#pragma unroll
    for (int q = 0; q < 2; ++q)
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const auto w = __builtin_amdgcn_permlane32_swap(__float_as_uint(s[u][q][j]), __float_as_uint(s[u][q][j + 4]),
                                                        false, false);
        s[u][q][j] = __uint_as_float(w[0]);
        s[u][q][j + 4] = __uint_as_float(w[1]);
      }
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const auto w = __builtin_amdgcn_permlane16_swap(__float_as_uint(s[u][0][j]), __float_as_uint(s[u][1][j]),
                                                      false, false);
      s[u][0][j] = __uint_as_float(w[0]);
      s[u][1][j] = __uint_as_float(w[1]);
    }
  }
}

// One output op without further operands (ACC, SILU, SWIGLU) over the wave's TM row
// subtiles: accumulator columns gn0 + u * jump .. + 8, gn0 the lane's own. TWO: the
// column subtiles are the two accumulators' same columns (the op's own is eo.a).
template <int OP, int TM, bool SUMSQ, bool TWO>
__device__ __forceinline__ void pp_epi(const GemmK& p, const EpiOutK& eo, int o2, const f32x16_t (&acc)[TM][2],
                                       const float* rsw, int64_t row_w, int gn0, int jump, int lane) {
  constexpr int NU = TWO ? 1 : 2;  // subtiles to store
  const bool sa = SUMSQ && ((p.rscale_mask >> eo.a) & 1u);
  const bool sb = SUMSQ && eo.b >= 0 && ((p.rscale_mask >> eo.b) & 1u);
  const int r_l = lane & 15;
  auto gcol = [&](int u) { return gn0 + u * jump; };
  // (windows are multiples of 8, gemm_pp_fits: an octet is wholly in or out)
  auto inside = [&](int u) { return gcol(u) >= eo.cb && gcol(u) < eo.ce; };
  const int nt = (int)min((p.M - row_w + 31) >> 5, (int64_t)TM);  // (the caller has checked row_w < M)
#pragma unroll 1
  for (int t = 0; t < nt; ++t) {
    // acc[t] to fixed registers, as octets
    float s[2][2][8];
#define TH_PP_TAKE(T_)                                                                                        \
  case T_:                                                                                                    \
    if constexpr (T_ < TM) {                                                                                  \
      _Pragma("unroll") for (int u = 0; u < 2; ++u)                                                           \
          _Pragma("unroll") for (int q = 0; q < 2; ++q)                                                       \
              _Pragma("unroll") for (int j = 0; j < 8; ++j) s[u][q][j] = acc[T_ < TM ? T_ : 0][u][8 * q + j]; \
    }                                                                                                         \
    break;
    switch (t) {
      TH_PP_TAKE(0)
      TH_PP_TAKE(1)
      TH_PP_TAKE(2)
      TH_PP_TAKE(3)
    }
#undef TH_PP_TAKE
    // The op is done here, so that it is done (and, for a bf16 output, rounded) before the
    // lanes trade.
    const float rr = SUMSQ && (sa || sb) ? rsw[32 * t + (lane & 31)] : 1.f;
#pragma unroll
    for (int q = 0; q < 2; ++q)
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        if constexpr (TWO) {  // own accumulator to s[0], by value
          const float x0 = s[0][q][e], x1 = s[1][q][e];
          float a = eo.a ? x1 : x0, bb = eo.b ? x1 : x0;
          if (sa) a *= rr;
          if (sb) bb *= rr;
          if constexpr (OP == TH_EPI_SILU) a = a * sigmoidf_(a);
          if constexpr (OP == TH_EPI_SWIGLU) a = a * sigmoidf_(a) * bb;
          s[0][q][e] = a;
        } else {
#pragma unroll
          for (int u = 0; u < 2; ++u) {
            float a = s[u][q][e];
            if (sa) a *= rr;
            if constexpr (OP == TH_EPI_SILU) a = a * sigmoidf_(a);
            s[u][q][e] = a;
          }
        }
      }
    if (o2 < 0 && eo.dtype == TH_BF16) {
      // packed pairs (trade_lanes on half the registers)
#pragma unroll
      for (int u = 0; u < NU; ++u) {
        uint32_t w[2][4];
#pragma unroll
        for (int q = 0; q < 2; ++q) {
#pragma unroll
          for (int k = 0; k < 4; ++k) w[q][k] = pk_bf16x2(s[u][q][2 * k], s[u][q][2 * k + 1]);
#pragma unroll
          for (int k = 0; k < 2; ++k) {
            const auto x = __builtin_amdgcn_permlane32_swap(w[q][k], w[q][k + 2], false, false);
            w[q][k] = x[0];
            w[q][k + 2] = x[1];
          }
        }
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          const auto x = __builtin_amdgcn_permlane16_swap(w[0][k], w[1][k], false, false);
          w[0][k] = x[0];
          w[1][k] = x[1];
        }
#pragma unroll
        for (int q = 0; q < 2; ++q) {
          const int64_t gm = row_w + 32 * t + 16 * q + r_l;
          if (gm < p.M && inside(u))
            *(uint4*)((uint16_t*)eo.ptr + gm * eo.ld + gcol(u) - eo.cb) = make_uint4(w[q][0], w[q][1], w[q][2], w[q][3]);
        }
      }
      continue;
    }
    trade_lanes<NU>(s);
#pragma unroll
    for (int u = 0; u < NU; ++u)
#pragma unroll
      for (int q = 0; q < 2; ++q) {
        const int64_t gm = row_w + 32 * t + 16 * q + r_l;
        if (gm < p.M && inside(u)) {
          const int64_t gc = gcol(u) - eo.cb;
          store8(eo.ptr, gm * eo.ld + gc, eo.dtype, true, 8, s[u][q]);
          if (o2 >= 0) {
            const EpiOutK& e2 = p.out[o2];
            store8(e2.ptr, gm * e2.ld + gc, e2.dtype, true, 8, s[u][q]);
          }
        }
      }
  }
}

// One output op with an operand per element over the wave's TM row subtiles, columns and
// TWO as in pp_epi: KIND 0 the extra operand (ADD, SOFTPLUS_ADD, MUL; XB: it is bf16),
// KIND 1 the RoPE tables (ROPE; TWO: ROPE_PAIR). What bounds it is the operand's latency:
// the octets of the next subtile (of its next 16 rows, with four loads per octet for the
// tables) are loaded before the present ones are stored, in code without branches around
// memory accesses, so that the wait for them leaves the stores in flight. (Loaded octet by
// octet behind the stores instead: residual 16384 x 1024 x 2048 64.9 us, now 62.0, 4096 rows 27.0,
// now 25.6; a residual in fp32 with bf16 and fp32 outputs and fused RoPE within 1% either way,
// there the stores and the tables' L2 reads bound it.)
template <int KIND, int TM, bool SUMSQ, bool TWO, bool XB, bool O2>
__device__ __forceinline__ void pp_epi_x(const GemmK& p, const EpiOutK& eo, const EpiOutK& e2, const f32x16_t (&acc)[TM][2],
                                         const float* rsw, int64_t row_w, int gn0, int jump, int lane) {
  constexpr int NU = TWO ? 1 : 2;                    // subtiles to store
  constexpr int NS = TWO && KIND == 0 ? 1 : 2;       // subtiles to trade
  constexpr int ES = XB ? 2 : 4;                     // bytes of an operand element
  constexpr int NX = KIND == 1 ? 4 : XB ? 1 : 2;     // 16-byte loads per octet
  const bool sa = SUMSQ && ((p.rscale_mask >> eo.a) & 1u);
  const bool sb = SUMSQ && eo.b >= 0 && ((p.rscale_mask >> eo.b) & 1u);
  const int r_l = lane & 15;
  const int rem = (int)min(p.M - row_w, (int64_t)32 * TM);  // rows of this wave
  // byte offsets of the lane's octets in row r_l of the wave's rows
  uint32_t vo[NU], v2[NU], vx[NU];
  const int os = eo.dtype == TH_BF16 ? 2 : 4, os2 = e2.dtype == TH_BF16 ? 2 : 4;
  const int ldx = KIND == 0 ? (int)p.ld_extra[eo.e] : 0;
#pragma unroll
  for (int u = 0; u < NU; ++u) {
    const int gc = gn0 + u * jump;
    const bool in = gc >= eo.cb && gc < eo.ce;  // (windows are multiples of 8: an octet is wholly in or out)
    vo[u] = in ? (uint32_t)((r_l * (int)eo.ld + gc - eo.cb) * os) : kNone;
    if constexpr (O2) v2[u] = in ? (uint32_t)((r_l * (int)e2.ld + gc - eo.cb) * os2) : kNone;
    if constexpr (KIND == 0) vx[u] = in ? (uint32_t)((r_l * ldx + gc - eo.cb) * ES) : kNone;
    else vx[u] = (uint32_t)(gc % p.hd) * 4;
  }
  const auto ro = wave_rows(eo.ptr, row_w * eo.ld * os);
  const auto r2 = wave_rows(e2.ptr, O2 ? row_w * e2.ld * os2 : 0);
  const auto rx = wave_rows(KIND == 0 ? p.extra[eo.e] : p.rcos, KIND == 0 ? row_w * ldx * ES : 0);
  const auto rt = wave_rows(KIND == 0 ? p.extra[eo.e] : p.rsin, 0);
  auto live = [&](uint32_t v, int row0) { return r_l < rem - row0 ? v : kNone; };

  // RoPE: table row of the lane's rows, stepped by 16 (one division a tile)
  uint32_t trow = 0;
  const uint32_t period = (uint32_t)p.period, step16 = KIND == 1 ? 16u % period : 0u;
  if constexpr (KIND == 1) trow = (uint32_t)(row_w + r_l) % period;
  constexpr int NQ = KIND == 0 ? 2 : 1;  // row halves loaded at a time
  u32x4_t x[NU][NQ][NX];
  auto fetch = [&](int row0) __attribute__((always_inline)) {  // rows row0 .. + 16 NQ
#pragma unroll
    for (int q = 0; q < NQ; ++q)
#pragma unroll
      for (int u = 0; u < NU; ++u) {
        if constexpr (KIND == 0) {
          const uint32_t v = live(vx[u], row0 + 16 * q);
          const int so = (row0 + 16 * q) * ldx * ES;
#pragma unroll
          for (int k = 0; k < NX; ++k) x[u][q][k] = __builtin_amdgcn_raw_buffer_load_b128(rx, v, so + 16 * k, 0);
        } else {
          const uint32_t v = trow * (uint32_t)p.hd * 4 + vx[u];
#pragma unroll
          for (int k = 0; k < 2; ++k) {
            x[u][q][k] = __builtin_amdgcn_raw_buffer_load_b128(rx, v, 16 * k, 0);
            x[u][q][2 + k] = __builtin_amdgcn_raw_buffer_load_b128(rt, v, 16 * k, 0);
          }
        }
      }
    if constexpr (KIND == 1) {
      trow += step16;
      trow = trow >= period ? trow - period : trow;
    }
  };
  // (The offset goes in through the lane's register alone: with a scalar register as the store's
  // own offset the compiler leaves out the wait between a 16-byte store and the next write of its
  // data registers, and the last lanes' data was overwritten on this chip.)
  auto put = [&](auto r, uint32_t v, int dtype, const float* f) __attribute__((always_inline)) {
    if (dtype == TH_BF16) {
      const u32x4_t w = {pk_bf16x2(f[0], f[1]), pk_bf16x2(f[2], f[3]), pk_bf16x2(f[4], f[5]), pk_bf16x2(f[6], f[7])};
      __builtin_amdgcn_raw_buffer_store_b128(w, r, v, 0, 0);
    } else {
#pragma unroll
      for (int k = 0; k < 2; ++k) {
        const u32x4_t w = {__float_as_uint(f[4 * k]), __float_as_uint(f[4 * k + 1]), __float_as_uint(f[4 * k + 2]),
                           __float_as_uint(f[4 * k + 3])};
        __builtin_amdgcn_raw_buffer_store_b128(w, r, v + 16 * k, 0, 0);
      }
    }
  };

  fetch(0);
#pragma unroll
  for (int t = 0; t < TM; ++t) {  // (subtiles past M: nothing is loaded or stored)
    float s[2][2][8];
    const float rr = SUMSQ && (sa || sb) ? rsw[32 * t + (lane & 31)] : 1.f;
#pragma unroll
    for (int q = 0; q < 2; ++q)
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const float x0 = acc[t][0][8 * q + e], x1 = acc[t][1][8 * q + e];
        float a = TWO && eo.a ? x1 : x0, b = TWO ? (eo.b ? x1 : x0) : x1;
        if (sa) a *= rr;
        if (TWO ? sb : sa) b *= rr;
        s[0][q][e] = a;
        s[1][q][e] = b;
      }
    trade_lanes<NS>(s);
#pragma unroll
    for (int q = 0; q < 2; ++q) {
      const int row0 = 32 * t + 16 * q;
      if constexpr (KIND == 0) {
#pragma unroll
        for (int u = 0; u < NU; ++u) {
          float xe[8];
#pragma unroll
          for (int k = 0; k < 4; ++k) {
            if constexpr (XB) {
              xe[2 * k] = __uint_as_float(x[u][q][0][k] << 16);
              xe[2 * k + 1] = __uint_as_float(x[u][q][0][k] & 0xffff0000u);
            } else {
              xe[k] = __uint_as_float(x[u][q][0][k]);
              xe[4 + k] = __uint_as_float(x[u][q][NX - 1][k]);
            }
          }
          float (&v)[8] = s[u][q];
          if (eo.op == TH_EPI_MUL) {
#pragma unroll
            for (int e = 0; e < 8; ++e) v[e] *= xe[e];
          } else {
#pragma unroll
            for (int e = 0; e < 8; ++e) v[e] += xe[e];
            // (a branch on the wave, not around memory accesses: a Mamba block's dt window is 16
            // columns of a tile, and 64 lanes' softplus of the subtile beside it cost 1 us)
            if (eo.op == TH_EPI_SOFTPLUS_ADD && __any(vo[u] != kNone)) {
#pragma unroll
              for (int e = 0; e < 8; ++e) v[e] = softplusf_(v[e]);
            }
          }
        }
        if (q == 0) continue;  // (both halves were loaded together)
      } else {
        // ROPE: the partner is the other subtile's same column. (The fma written out: left to
        // contraction, which product it rounds could differ between two outputs of one value.)
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          const float a = s[0][q][e], b = s[1][q][e];
          const int k = e >> 2, w = e & 3;
          s[0][q][e] = fmaf(a, __uint_as_float(x[0][0][k][w]), (TWO ? b : -b) * __uint_as_float(x[0][0][2 + k][w]));
          if constexpr (!TWO)
            s[1][q][e] = fmaf(b, __uint_as_float(x[NU - 1][0][k][w]), a * __uint_as_float(x[NU - 1][0][2 + k][w]));
        }
      }
      if (row0 + 16 < 32 * TM) fetch(row0 + 16);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int h = NQ == 2 ? 0 : q; h <= q; ++h)
#pragma unroll
        for (int u = 0; u < NU; ++u) {
          const int rs = 32 * t + 16 * h;
          put(ro, live(vo[u] + rs * (int)eo.ld * os, rs), eo.dtype, s[u][h]);
          if constexpr (O2) put(r2, live(v2[u] + rs * (int)e2.ld * os2, rs), e2.dtype, s[u][h]);
        }
      __builtin_amdgcn_sched_barrier(0);
    }
  }
}

}  // namespace

// p.asplit (two accumulators): waves wn = 0, 1 hold accumulator 0, waves 2, 3
// accumulator 1 (64 columns each) instead of 32 columns of both.
template <int TM, bool SUMSQ, int NACC>
__global__ void __launch_bounds__(512, 1) gemm_bf16_pp_kernel(GemmK p) {
#if defined(__HIP_DEVICE_COMPILE__)
  static_assert(TM >= 2 && TM <= 4 && (NACC == 1 || NACC == 2), "tile shape");
  constexpr int T0 = (TM + 1) / 2, T1 = TM - T0;  // row subtiles of A0 and A1
  constexpr int BM = 64 * TM, WM = 32 * TM;
  constexpr int bn = 256 / NACC;
  constexpr int ASTAGE = BM * 128, BSTAGE = 256 * 128;  // bytes of one 64-deep stage
  constexpr int BBASE = 2 * ASTAGE;
  constexpr int MAIN = 2 * (ASTAGE + BSTAGE);
  __shared__ __attribute__((aligned(16))) char smem[MAIN + BM * 4];
  float* rsx = (float*)(smem + MAIN);  // row scales of the current tile row

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave >> 2, wn = wave & 3;
  const int tiles = p.tiles_m * p.tiles_n;
  // K steps, an even number: all but the last two are whole, and the chunks (8
  // columns) left for those two are the last v1 and v2 of their 64 columns.
  const int nk = 2 * (int)((p.K + 127) >> 7);
  const int krest = (int)(p.K >> 3) - 8 * (nk - 2), v2 = min(krest, 8), v1 = krest - v2;

  // Column of the wave's (and, for the loads, of N-wave w's) first subtile
  // within an accumulator's tile, and the distance to the second one.
  const bool split = NACC == 2 && p.asplit;
  const int half = p.pair_hd >> 1;
  const int jump = half >= 32 ? half : 32;
  auto col0_of = [&](int w) {
    if (NACC == 2 && !split) return 32 * w;
    const int blk = NACC == 2 ? w & 1 : w;
    if (half < 32) return 64 * blk;
    const int nb = half >> 5, head = blk / nb;
    return head * p.pair_hd + (blk - head * nb) * 32;
  };
  // LDS row (packed rhs row within the tile) of subtile u of N-wave w
  auto brow_of = [&](int w, int u) {
    if (NACC == 2 && !split) return u * bn + 32 * w;
    return (NACC == 2 ? (w >> 1) * bn : 0) + col0_of(w) + u * jump;
  };

  // LDS rows are 128 bytes (64 bf16), chunk c of row R in slot c ^ g(R), g(R) =
  // (R & 7) ^ ((R >> 3) & 1). Loads fill 8 rows (1 KB) each.
  // lhs: region A0 is rows wm' WM + 0 .. 32 T0 of both row halves, A1 the rest.
  // Wave w loads 4 T0 (4 T1) rows of row half w / 4 as T0 (T1) loads of 8 rows:
  // load i of region h is rows (w / 4) WM + 32 T0 h + 8 (i 4 + w % 4).
  auto arow = [&](int h, int i) { return (wave >> 2) * WM + 32 * T0 * h + 8 * (4 * i + (wave & 3)); };
  uint32_t voa[TM];
  // rhs: region B0 (B1) is subtile 0 (1) of the four N-waves, 128 rows; wave w
  // loads rows 16 (w % 2) .. + 16 of N-wave w / 2's subtile, as two loads of 8 rows.
  const int br0 = brow_of(wave >> 1, 0) + 16 * (wave & 1), br1 = brow_of(wave >> 1, 1) + 16 * (wave & 1);
  uint32_t vob0, vob1;
  const uint32_t lds0 = (uint32_t)(uintptr_t)smem;

  const char *ga = nullptr, *gb0 = nullptr, *gb1 = nullptr;
  // Per-lane load offsets of tile row tm: set for the first loads of a tile, and with 256
  // rows again at the head of its K loop, so that the epilogue between need not keep them.
  auto lane_offsets = [&](int tm) __attribute__((always_inline)) {
    const int arows = (int)min((int64_t)BM, p.M - (int64_t)tm * BM);  // rows past M re-read row M - 1 (never stored)
    const int l = fresh_lane(), lr = l >> 3;
    const uint32_t c0 = (uint32_t)(((l & 7) ^ lr) << 4);
    vob0 = (uint32_t)(lr * p.ldb * 2) + c0;  // rows at an even multiple of 8
    vob1 = (uint32_t)((8 + lr) * p.ldb * 2) + (c0 ^ 16u);
#pragma unroll
    for (int i = 0; i < TM; ++i) {
      const int r = i < T0 ? arow(0, i) : arow(1, i - T0);
      voa[i] = (uint32_t)(min(r + lr, arows - 1) * p.lda * 2) + ((r >> 3) & 1 ? c0 ^ 16u : c0);
    }
  };
  auto tile_rsrc = [&](int L, int& tm, int& tn) {
    pp_map(L, p.tiles_m, p.tiles_n, tm, tn);
    ga = (const char*)p.A + (int64_t)tm * BM * p.lda * 2;
    const char* gb = (const char*)p.B + (int64_t)tn * 256 * p.ldb * 2;
    gb0 = gb + (int64_t)br0 * p.ldb * 2;
    gb1 = gb + (int64_t)br1 * p.ldb * 2;
    lane_offsets(tm);
  };
  const int64_t k1 = (p.K - 8 * v2 - 64) * 2, k2 = (p.K - 64) * 2;
  auto kofs = [&](int kt) { return kt < nk - 2 ? (int64_t)kt * 128 : kt == nk - 2 ? k1 : k2; };
  auto load_a = [&](auto hc, int kt, int st) __attribute__((always_inline)) {
    constexpr int H = decltype(hc)::value;
    const char* g = ga + kofs(kt);
#pragma unroll
    for (int i = 0; i < (H ? T1 : T0); ++i)
      dma_load16(g, voa[H ? T0 + i : i], lds0 + st * ASTAGE + arow(H, i) * 128);
  };
  auto load_b = [&](int u, int kt, int st) __attribute__((always_inline)) {
    const char* g = (u ? gb1 : gb0) + kofs(kt);
    const uint32_t d = lds0 + BBASE + st * BSTAGE + (u ? br1 : br0) * 128;
    dma_load16(g, vob0, d);
    dma_load16(g, vob1, d + 1024);
  };
  using C0 = std::integral_constant<int, 0>;
  using C1 = std::integral_constant<int, 1>;

  // fragment addresses: per 16-deep step ks, chunk 2 ks + lane / 32
  int fch[4], abase, bbase0, bbase1;
  auto lane_fragments = [&]() __attribute__((always_inline)) {
    const int l = fresh_lane();
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) fch[ks] = ((ks * 2 + (l >> 5)) ^ (l & 7) ^ ((l >> 3) & 1)) << 4;
    abase = (wm * WM + (l & 31)) * 128;
    bbase0 = BBASE + (brow_of(wn, 0) + (l & 31)) * 128;
    bbase1 = BBASE + (brow_of(wn, 1) + (l & 31)) * 128;
  };

  bf16x8_t fa[T0][4], fb[2][4];
  f32x16_t acc[TM][2];
  const uint32_t odd = wn & 1 ? ~0u : 0u;
  // Row sums of squares of subtile t = wn, as four chains (a dependent v_dot2
  // waits for the one before). Only where a workgroup's tile row changes: its
  // tiles walk down the columns of eight tile rows, mostly along one row, and
  // the scales stay in LDS.
  float ss[4];
  bool new_row = SUMSQ, need_ss = SUMSQ && p.rs_parts == nullptr;
  const bf16x8_t zero8 = {};
  auto read_a = [&](auto hc, int st) __attribute__((always_inline)) {
    constexpr int H = decltype(hc)::value;
#pragma unroll
    for (int ks = 0; ks < 4; ++ks)
#pragma unroll
      for (int t = 0; t < (H ? T1 : T0); ++t)
        fa[t][ks] = *(const bf16x8_t*)(smem + abase + fch[ks] + st * ASTAGE + (H * T0 + t) * 4096);
  };
  auto read_b = [&](bf16x8_t (&f)[4], int base, int st) __attribute__((always_inline)) {
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) f[ks] = *(const bf16x8_t*)(smem + base + fch[ks] + st * BSTAGE);
  };
  // zero all but the last v chunks of a partial step's fragments
  auto mask4 = [&](bf16x8_t (&f)[4], int v) __attribute__((always_inline)) {
#pragma unroll
    for (int ks = 0; ks < 4; ++ks)
      if (2 * ks + (lane >> 5) < 8 - v) f[ks] = zero8;
  };
  // (keeps what follows a conditional mask from being computed in both of its
  // branches, which cost a second set of fragment registers)
  auto pin4 = [&](bf16x8_t (&f)[4]) __attribute__((always_inline)) {
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) asm volatile("" : "+v"(f[ks]));
  };
  auto mfmas = [&](auto hc, int u, const bf16x8_t (&f)[4]) __attribute__((always_inline)) {
    constexpr int H = decltype(hc)::value;
    __builtin_amdgcn_s_setprio(1);
#pragma unroll
    for (int ks = 0; ks < 4; ++ks)
#pragma unroll
      for (int t = 0; t < (H ? T1 : T0); ++t)
        acc[H * T0 + t][u] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(f[ks], fa[t][ks], acc[H * T0 + t][u], 0, 0, 0);
    __builtin_amdgcn_s_setprio(0);
    __builtin_amdgcn_sched_barrier(0);
  };
  // Row sums of squares of half H's subtile that this wave owns (t = wn), in the
  // memory part of the half's second phase: under the other group's MFMAs.
  auto sumsq_half = [&](auto hc) __attribute__((always_inline)) {
    constexpr int H = decltype(hc)::value, TH = H ? T1 : T0;
    if constexpr (SUMSQ) {
      if (need_ss && (H ? wn >= T0 && wn < TM : wn < T0)) {
#pragma unroll
        for (int ks = 0; ks < 4; ++ks) {
          // (a select of values, word by word: of array elements it would be one of
          // addresses, and the fragments would live in scratch memory)
          const u32x4_t x0 = __builtin_bit_cast(u32x4_t, fa[0][ks]), x1 = __builtin_bit_cast(u32x4_t, fa[TH - 1][ks]);
          u32x4_t x = x0;
          if constexpr (TH > 1) {
#pragma unroll
            for (int i = 0; i < 4; ++i) x[i] = (x0[i] & ~odd) | (x1[i] & odd);
          }
          typedef __bf16 b2_t __attribute__((ext_vector_type(2)));
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const b2_t w = __builtin_bit_cast(b2_t, (uint32_t)x[i]);
            ss[i] = __builtin_amdgcn_fdot2_f32_bf16(w, w, ss[i], false);
          }
          __builtin_amdgcn_sched_barrier(0);
        }
      }
    }
  };
  // the end of a phase's memory part and of its MFMA part
  auto mem_end = [&]() __attribute__((always_inline)) {
    wait_lgkmcnt0();
    barrier_keep_loads();
    __builtin_amdgcn_sched_barrier(0);
  };
  auto mfma_end = [&]() __attribute__((always_inline)) {
    barrier_keep_loads();
    __builtin_amdgcn_sched_barrier(0);
  };

  // One K step in stage PAR. MODE 0: steady (loads of step kt + 2 go out);
  // 1: the last step but one, 2: the last one (no loads; the waits count what
  // is still in flight). Loads go out as B0 2, A0 T0, B1 2, A1 T1 per step.
  auto kstep = [&](int kt, auto parc, auto modec) __attribute__((always_inline)) {
    constexpr int PAR = decltype(parc)::value, MODE = decltype(modec)::value;
    constexpr int NS = 4 + TM;  // loads per K step
    const int v = MODE == 1 ? v1 : v2;  // valid chunks of the last two steps
    auto& b0 = fb[PAR];
    auto& b1 = fb[PAR ^ 1];
    // phase 0
    read_a(C0{}, PAR);
    if constexpr (MODE == 0) {
      load_b(0, kt + 2, PAR);
      wait_vmcnt<NS + T1 + 2>();  // B1(kt)
    } else if constexpr (MODE == 1) {
      wait_vmcnt<NS + T1>();
    } else {
      wait_vmcnt<T1>();
    }
    if (MODE != 0 && v < 8) {
      wait_lgkmcnt0();
      mask4(b0, v);
#pragma unroll
      for (int t = 0; t < T0; ++t) mask4(fa[t], v);
    }
    if constexpr (MODE != 0) {
#pragma unroll
      for (int t = 0; t < T0; ++t) pin4(fa[t]);
    }
    mem_end();
    mfmas(C0{}, 0, b0);
    mfma_end();
    // phase 1
    read_b(b1, bbase1, PAR);
    if constexpr (MODE == 0) {
      load_a(C0{}, kt + 2, PAR);
      wait_vmcnt<NS + 2 + T0>();  // A1(kt)
    } else if constexpr (MODE == 1) {
      wait_vmcnt<NS>();
    } else {
      wait_vmcnt<0>();
    }
    sumsq_half(C0{});
    if (MODE != 0 && v < 8) {
      wait_lgkmcnt0();
      mask4(b1, v);
    }
    mem_end();
    mfmas(C0{}, 1, b1);
    mfma_end();
    // phase 2
    read_a(C1{}, PAR);
    if constexpr (MODE == 0) {
      load_b(1, kt + 2, PAR);
      wait_vmcnt<NS + T0 + 2>();  // B0(kt + 1)
    } else if constexpr (MODE == 1) {
      wait_vmcnt<NS - 2>();
    }
    if (MODE != 0 && v < 8) {
      wait_lgkmcnt0();
#pragma unroll
      for (int t = 0; t < T1; ++t) mask4(fa[t], v);
    }
    if constexpr (MODE != 0) {
#pragma unroll
      for (int t = 0; t < T1; ++t) pin4(fa[t]);
    }
    mem_end();
    mfmas(C1{}, 1, b1);
    mfma_end();
    // phase 3
    if constexpr (MODE != 2) read_b(b1, bbase0, PAR ^ 1);
    if constexpr (MODE == 0) {
      load_a(C1{}, kt + 2, PAR);
      wait_vmcnt<NS + 2 + T1>();  // A0(kt + 1)
    } else if constexpr (MODE == 1) {
      wait_vmcnt<2 + T1>();
    }
    sumsq_half(C1{});
    mem_end();
    mfmas(C1{}, 0, b0);
  };
  using M0 = std::integral_constant<int, 0>;
  using M1 = std::integral_constant<int, 1>;
  using M2 = std::integral_constant<int, 2>;

  auto start_tile = [&]() __attribute__((always_inline)) {
#pragma unroll
    for (int kt = 0; kt < 2; ++kt) {
      load_b(0, kt, kt);
      load_a(C0{}, kt, kt);
      load_b(1, kt, kt);
      load_a(C1{}, kt, kt);
    }
  };

  int L = blockIdx.x;
  if (L >= tiles) return;
  int tmi, tni;
  // scale of the tile row's row r, whose own sum of squares is `own` (unless the producer's parts are given)
  auto row_scale = [&](int r, float own) __attribute__((always_inline)) {
    const int64_t gr = (int64_t)tmi * BM + r;
    const float v = row_sumsq(p, gr, own);
    rsx[r] = rsqrtf(v * p.inv_k + p.eps);
    if (p.sumsq_out && gr < p.M) p.sumsq_out[gr] = v;  // (every workgroup of the row writes the same value)
  };
  tile_rsrc(L, tmi, tni);
  start_tile();
  if constexpr (TM < 4) lane_fragments();

  for (;;) {
    if constexpr (TM == 4) {
      // (pinned here, where the tile's first loads are in flight: the compiler would compute the
      // offsets past the barrier, 0.3 us of a tile)
      lane_offsets(tmi);
      lane_fragments();
      asm volatile("" : "+v"(vob0), "+v"(vob1), "+v"(abase), "+v"(bbase0), "+v"(bbase1));
#pragma unroll
      for (int i = 0; i < TM; ++i) asm volatile("" : "+v"(voa[i]));
#pragma unroll
      for (int ks = 0; ks < 4; ++ks) asm volatile("" : "+v"(fch[ks]));
    }
    // B0(0) and A0(0) have landed everywhere, then the first B fragments
    wait_vmcnt<4 + TM + 2 + T1>();
    barrier_keep_loads();
    read_b(fb[0], bbase0, 0);
    ss[0] = ss[1] = ss[2] = ss[3] = 0.f;
#pragma unroll
    for (int t = 0; t < TM; ++t)
#pragma unroll
      for (int u = 0; u < 2; ++u)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[t][u][r] = 0.f;
    if constexpr (SUMSQ) {
      // Row scales from the producer's partial sums: here, where the tile's first loads are in
      // flight (after the K loop nothing is, and every wave waits), and past the barrier behind
      // which no wave reads the last tile row's scales.
      if (new_row && p.rs_parts != nullptr && wn < TM) {
        const int r = fresh_lane();
        if (r < 32) row_scale(wm * WM + 32 * wn + r, 0.f);
      }
    }
    mem_end();
    if (wm) mfma_end();  // the half-phase offset of the second group

    for (int kt = 0; kt < nk - 2; kt += 2) {
      kstep(kt, C0{}, M0{});
      mfma_end();
      kstep(kt + 1, C1{}, M0{});
      mfma_end();
    }
    kstep(nk - 2, C0{}, M1{});
    mfma_end();
    kstep(nk - 1, C1{}, M2{});
    if constexpr (SUMSQ) {
      const float own = (ss[0] + ss[1]) + (ss[2] + ss[3]);
      const float v = own + __shfl_xor(own, 32);
      if (need_ss && wn < TM && lane < 32) row_scale(wm * WM + 32 * wn + lane, v);
    }
    wait_lgkmcnt0();
    mfma_end();
    if (!wm) mfma_end();  // both groups are level again, past every read of the stages

    const int Ln = L + (int)gridDim.x;
    const bool more = Ln < tiles;
    const int64_t row_w = (int64_t)tmi * BM + wm * WM;
    const int64_t col_t = (int64_t)tni * bn;
    int tmn = 0, tnn = 0;
    if (more) {
      tile_rsrc(Ln, tmn, tnn);
      start_tile();
    }

    // ---- epilogue: registers only
    const GemmK& pe = fresh_args();
    const int le = fresh_lane();
    const int c0 = col0_of(wn);
    const int gn0 = (int)col_t + c0 + 8 * ((le >> 5) + 2 * ((le >> 4) & 1));  // the lane's octet of a subtile
    const int lo = (int)col_t + c0, hi = lo + (NACC == 2 && !split ? 32 : jump + 32);
    const float* rsw = rsx + wm * WM;
    const int n_out = row_w < pe.M ? pe.n_out : 0;  // (a wave wholly past the last row has nothing to do)
    for (int o = 0; o < n_out; ++o) {
      const EpiOutK& eo = pe.out[o];
      // an fp32 copy right after its bf16 output is stored from the same values
      const int o2 = o + 1 < n_out && same_values(eo, pe.out[o + 1]) ? o + 1 : -1;
      if (o2 >= 0) ++o;
      if (split && eo.a != (wn >> 1)) continue;
      if (eo.ce <= lo || eo.cb >= hi) continue;  // nothing of it in this wave
#define TH_PP_CASE(OP_, TWO_)                                               \
  pp_epi<OP_, TM, SUMSQ, TWO_>(pe, eo, o2, acc, rsw, row_w, gn0, jump, le); \
  break
#define TH_PP_X(KIND_, TWO_, XB_)                                                                          \
  if (o2 >= 0)                                                                                             \
    pp_epi_x<KIND_, TM, SUMSQ, TWO_, XB_, true>(pe, eo, pe.out[o2], acc, rsw, row_w, gn0, jump, le); \
  else                                                                                                     \
    pp_epi_x<KIND_, TM, SUMSQ, TWO_, XB_, false>(pe, eo, eo, acc, rsw, row_w, gn0, jump, le)
      if (NACC == 1 || split) {
        switch (eo.op) {
          case TH_EPI_ACC: TH_PP_CASE(TH_EPI_ACC, false);
          case TH_EPI_SILU: TH_PP_CASE(TH_EPI_SILU, false);
          case TH_EPI_ROPE: TH_PP_X(1, false, false); break;
          default:
            if (pe.extra_dtype[eo.e] == TH_BF16) { TH_PP_X(0, false, true); } else { TH_PP_X(0, false, false); }
        }
      } else if constexpr (NACC == 2) {
        switch (eo.op) {
          case TH_EPI_ACC: TH_PP_CASE(TH_EPI_ACC, true);
          case TH_EPI_SILU: TH_PP_CASE(TH_EPI_SILU, true);
          case TH_EPI_SWIGLU: TH_PP_CASE(TH_EPI_SWIGLU, true);
          case TH_EPI_ROPE_PAIR: TH_PP_X(1, true, false); break;
          default:
            if (pe.extra_dtype[eo.e] == TH_BF16) { TH_PP_X(0, true, true); } else { TH_PP_X(0, true, false); }
        }
      }
#undef TH_PP_X
#undef TH_PP_CASE
    }
    if (!more) break;
    L = Ln;
    new_row = SUMSQ && tmn != tmi;
    need_ss = new_row && p.rs_parts == nullptr;
    tmi = tmn;
    tni = tnn;
  }
#endif
}

// Operand and output forms the kernel covers (th_gemm has checked the rest).
bool gemm_pp_fits(const GemmK& k) {
  if (k.K < 128 || k.M >= ((int64_t)1 << 31) || k.N >= ((int64_t)1 << 31)) return false;
  constexpr int64_t two_gib = (int64_t)1 << 31;
  auto rows_fit = [](int64_t ld, int bytes) { return ld < two_gib / (256 * bytes); };
  if (!rows_fit(k.lda, 2) || !rows_fit(k.ldb, 2)) return false;
  if (!((k.n_acc == 1 && k.bn == 256) || (k.n_acc == 2 && k.bn == 128))) return false;
  bool rope = false, pair = false;
  for (int o = 0; o < k.n_out; ++o) {
    rope |= k.out[o].op == TH_EPI_ROPE;
    pair |= k.out[o].b >= 0;
    // whole aligned octets in every output and operand row, a tile's rows within 2 GiB
    if (!k.out[o].vec8 || k.out[o].ce % 8 != 0 || !rows_fit(k.out[o].ld, 4)) return false;
    if (k.out[o].e >= 0 && (!k.extra_vec8[k.out[o].e] || !rows_fit(k.ld_extra[k.out[o].e], 4))) return false;
    if ((k.out[o].op == TH_EPI_ROPE || k.out[o].op == TH_EPI_ROPE_PAIR) && (int64_t)k.period * k.hd * 4 >= two_gib) return false;
  }
  // fused RoPE: heads of 64 and wider, whose partners meet in a wave (narrower
  // ones would need columns of other lanes); two accumulators: whole-accumulator
  // waves, and those no op of two accumulators
  if (rope && k.hd < 64) return false;
  if (k.n_acc == 1) return !pair && (!rope || 256 % k.hd == 0);
  return !rope || (128 % k.hd == 0 && !pair);
}

// Rows of the tile: the choice of 256, 192 and 128 with the smallest estimate (us, in
// *us) of rounds * (K steps * per-step time + per-tile time), the K steps an even number.
// A step's time grows with the share of the CUs at work, and by another 0.1 us once they are
// at work for long (the clock falls: 256-row steps measured 0.94 us on 4 CUs, 1.25 on 192,
// 1.45 - 1.6 on all 256; 192-row steps 0.75, 0.82 at half, 1.1 - 1.2; 128-row steps 0.47, 0.68
// at three quarters, 0.75 - 0.93). Own sums of squares cost 0.14 us a step where a
// workgroup's tile row is new, rotated tiles 6 us, a residual in fp32 2 to 10 us.
// The constants here and in bf16_loop_us (gemm.hip) are fitted to what the choice among the
// loops loses over 2125 shapes, each loop timed on each (32 .. 16384 rows, K = 128 .. 14336,
// N = 256 .. 50280, eight kinds of outputs, sizes drawn as well as round): 0.4% of the time
// on average; 0.7% over 467 drawn shapes that the fit has not seen.
int gemm_pp_rows(const GemmK& k, const EpiCost& ec, int64_t cus, double* us) {
  static const struct { int bm; double c0, c1, e; } shape[] = {
      {256, 0.868, 0.570, 12.0}, {192, 0.611, 0.454, 9.91}, {128, 0.465, 0.243, 8.14}};
  const double nk = 2.0 * (double)cdiv(k.K, 128);
  const double own_ss = k.sumsq && k.rs_parts == nullptr ? 0.137 * nk : 0;
  int best = 256;
  *us = 1e30;
  for (const auto& c : shape) {
    const int64_t tiles = cdiv(k.M, c.bm) * k.tiles_n, rounds = cdiv(tiles, cus);
    const double fill = (double)tiles / (double)(rounds * cus);
    const double step = c.c0 + fill * (c.c1 + 0.107 * std::min(1.0, (double)rounds * nk / 256));
    const double epi = ec.wide * (0.891 + 4.17 * fill) + 6.06 * ec.rope + 0.384 * (ec.outs - 1);
    const double t = (double)rounds * (nk * step + c.e + epi) + own_ss;
    if (t < *us) {
      *us = t;
      best = c.bm;
    }
  }
  return best;
}

template <int TM, int NACC>
static void launch_pp(const GemmK& k, int grid, hipStream_t s) {
  if (k.sumsq)
    hipLaunchKernelGGL((gemm_bf16_pp_kernel<TM, true, NACC>), dim3(grid), dim3(512), 0, s, k);
  else
    hipLaunchKernelGGL((gemm_bf16_pp_kernel<TM, false, NACC>), dim3(grid), dim3(512), 0, s, k);
}

int launch_gemm_pp(const GemmK& k0, int bm, hipStream_t s) {
  GemmK k = k0;
  bool rope = false;
  for (int o = 0; o < k.n_out; ++o) rope |= k.out[o].op == TH_EPI_ROPE;
  k.pair_hd = rope && k.hd >= 64 ? k.hd : 0;
  k.asplit = k.n_acc == 2 && k.pair_hd ? 1 : 0;
  k.tiles_m = (int)cdiv(k.M, bm);
  const int64_t tiles = (int64_t)k.tiles_m * k.tiles_n;
  const int cus = device_cus() > 0 ? device_cus() : 256;
  const int grid = (int)(tiles < cus ? tiles : cus);
  if (k.n_acc == 1) {
    switch (bm) {
      case 128: launch_pp<2, 1>(k, grid, s); break;
      case 192: launch_pp<3, 1>(k, grid, s); break;
      default: launch_pp<4, 1>(k, grid, s); break;
    }
  } else {
    switch (bm) {
      case 128: launch_pp<2, 2>(k, grid, s); break;
      case 192: launch_pp<3, 2>(k, grid, s); break;
      default: launch_pp<4, 2>(k, grid, s); break;
    }
  }
  TH_CHECK_LAUNCH();
  return TH_OK;
}

}  // namespace th
