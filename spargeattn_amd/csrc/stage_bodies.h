// Device code of the stages in front of the attention kernel, as bodies that more than one kernel is built from: the
// stage-by-stage entry points launch one body per kernel (maskpred.hip, vquant.hip), the whole-operator entry point
// launches several independent ones side by side in one kernel (forward.hip).  A body takes its place in the problem
// (block, head) as arguments and its LDS as a pointer, so that bodies sharing a kernel share one allocation.
//
// Include only in translation units compiled with -ffp-contract=off (see the arithmetic contract in maskpred.hip).
#pragma once
#include "common.h"
#include "launch.h"

#include <type_traits>

namespace spg {

// =============================================================================================
// K column mean
// =============================================================================================
template <int D, int NT = 256> constexpr int km_partial_lds() { return NT / (D / 8) * D * 8; }
template <int D, int DT, int NT = 256>
__device__ __forceinline__ void km_partial_body(const uint16_t *__restrict__ k, const Strides &ks, int H,
                                                double *__restrict__ part, int N, int rows_per_chunk, int chunk, int nchunk,
                                                int bh, unsigned char *smem) {
  constexpr int TPR = D / 8;      // lanes per row (16 B each)
  constexpr int RPP = NT / TPR;   // rows per pass of the workgroup
  const int c = threadIdx.x % TPR, r = threadIdx.x / TPR;
  const int row0 = chunk * rows_per_chunk;
  const int row1 = min(N, row0 + rows_per_chunk);
  const uint16_t *base = k + (size_t)(bh / H) * ks.sb + (size_t)(bh % H) * ks.sh + c * 8;
  double acc[8];
#pragma unroll
  for (int e = 0; e < 8; e++) acc[e] = 0.0;
#pragma unroll 4
  for (int row = row0 + r; row < row1; row += RPP) {
    const uint4 v = load_stream_u4(base + (size_t)row * ks.sn);
    const uint32_t w[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
    for (int e = 0; e < 4; e++) {
      acc[2 * e] += (double)elem_to_f32<DT>((uint16_t)(w[e] & 0xffffu));
      acc[2 * e + 1] += (double)elem_to_f32<DT>((uint16_t)(w[e] >> 16));
    }
  }
  double(*sm)[D] = (double(*)[D])smem;
#pragma unroll
  for (int e = 0; e < 8; e++) sm[r][c * 8 + e] = acc[e];
  __syncthreads();
  if (threadIdx.x < D) {
    double s = 0.0;
    for (int i = 0; i < RPP; i++) s += sm[i][threadIdx.x];
    part[((size_t)bh * nchunk + chunk) * D + threadIdx.x] = s;
  }
}

// =============================================================================================
// pool + sim + INT8 quantisation.  One workgroup per (block, b*h).
// =============================================================================================
// IEEE binary32 quotient a/b with a reciprocal shared by many numerators: r = RN(1/b) (one correctly rounded
// division), then q = RN(a*r), one exact residual and one correction (Markstein).  div_selftest_kernel below
// compares it with the hardware's correctly rounded division for every finite binary16/bfloat16 numerator with
// |a| >= 2^-100 against pseudo-random divisors: the only difference is the sign of a zero quotient, which no user of
// the result can see.
// Valid while b stays in [2^-60, 2^60] (no scaling of the operands is done); quotients below 2^-100 in magnitude
// may be off in the last place, far below anything the callers resolve.
__device__ __forceinline__ float exact_rcp(float b) { return 1.0f / b; }
__device__ __forceinline__ float div_by(float a, float b, float r) {
  const float q = a * r;
  const float e = __builtin_fmaf(-b, q, a);
  return __builtin_fmaf(e, r, q);
}
constexpr float CODE_MAGIC = 12582912.0f;   // 1.5 * 2^23
// The INT8 code of an element a under scale s is trunc(RN(RN(a / s) + 0.5)) with the sign of a.
__device__ __forceinline__ float away_from_zero(float quotient) { return quotient + __builtin_copysignf(0.5f, quotient); }
// That is the quotient to the nearest integer, unless it comes so close to n + 1/2 that one of the roundings decides: the quotient is off by at
// most 2^-24 of itself, the sum by 2^-24 (n + 1).  Rounding a * m once to an integer (an fma onto 1.5 2^23), with m = r = RN(1 / s), off by 2^-24,
// or the float above it, off by 3 2^-24 at most, gives the same code for every a with |a / s - (n + 1/2)| > 3 2^-24 (n + 1/2) for all n.  The
// others lie within 2^-22 and a little of t = RN((n + 1/2) s), and 16-bit floats are 2^-11 of themselves or more apart: of the elements up
// to the block's maximum, for which n ends at 126, one for each n can be in doubt, the one next to t.  So all of them are decided at
// once, two n per lane, by working out both codes of that element.  Returns an m that gives the codes of the division, r where it does, or 0 if
// neither does.
//
// Counted over every maximum from 10^-3 to the formats' top: r gives the codes for 99 to 100 % of those below 100.  Above, where the 1e-7 in s
// is lost, half the maximum is a tie, 63.5 s, that the rounding of r decides: r gives them for 55 to 65 % of the maxima, the float above it for 86
// to 96, one of the two for 98 to 99 %.  The stages in front are bound by their vector instructions as much as by memory: 2.75
// instructions per element for its code instead of 7.  us per call with divisions / as here, maxima of Q and K of 50 to 100: mask H48 N16384 Nk1000
// 184.8 / 172.9, FP16 PV H24 N8192 causal 287.0 / 280.8, H16 Nq8190 Nk2500 fp16 with per-warp scales 106.5 / 102.5, GQA 32/8 N4096 100.2 /
// 97.6, H30 N8192 D64 279.9 / 275.0, H2 N4096 43.3 / 42.7; of 400 to 800 186.3 / 173.5, 283.2 / 278.2, 107.4 / 103.3, 100.1 / 97.7, 276.7 / 273.3, 43.4 / 42.9.
template <int DT> __device__ __forceinline__ float code_multiplier(float s, float r) {
#pragma clang fp contract(off)
  const float n0 = (float)(threadIdx.x & 63) + 0.5f;
  auto differs = [&](float m) {
    bool any = false;
#pragma unroll
    for (int i = 0; i < 2; i++) {
      const float t = (i == 0 ? n0 : fminf(n0 + 64.f, 126.5f)) * s;
      const float a = elem_to_f32<DT>(f32_to_elem<DT>(t));   // the element next to t
      const uint16_t code = (uint16_t)(uint32_t)(div_by(a, s, r) + 0.5f);
      any |= (uint16_t)__builtin_bit_cast(uint32_t, __builtin_fmaf(a, m, CODE_MAGIC)) != code;   // (CODE_MAGIC ends in 22 zero bits)
    }
    return __any(any) != 0;
  };
  if (!differs(r)) return r;
  const float above = __builtin_bit_cast(float, __builtin_bit_cast(int, r) + 1);
  return !differs(above) ? above : 0.f;
}
// four floats CODE_MAGIC + code -> the four codes
__device__ __forceinline__ uint32_t pack_codes(float v0, float v1, float v2, float v3) {
  const uint32_t b0 = __builtin_bit_cast(uint32_t, v0), b1 = __builtin_bit_cast(uint32_t, v1);
  const uint32_t b2 = __builtin_bit_cast(uint32_t, v2), b3 = __builtin_bit_cast(uint32_t, v3);
  return __builtin_amdgcn_perm(__builtin_amdgcn_perm(b3, b2, 0x0c0c0400u), __builtin_amdgcn_perm(b1, b0, 0x0c0c0400u), 0x05040100u);
}
__device__ __forceinline__ bool rcp_safe(float b) { return b >= 0x1p-60f && b <= 0x1p60f; }

// Packed 16-bit helpers.  A tile is kept in registers as the 16-bit patterns it was loaded with (two per register) and
// widened where it is used: half the registers of a binary32 copy, which is what lets enough workgroups share a CU to
// keep HBM busy.
typedef unsigned short u16x2_t __attribute__((ext_vector_type(2)));
__device__ __forceinline__ uint32_t pk_max_u16(uint32_t a, uint32_t b) {
  return __builtin_bit_cast(uint32_t, __builtin_elementwise_max(__builtin_bit_cast(u16x2_t, a), __builtin_bit_cast(u16x2_t, b)));
}
template <int DT> __device__ __forceinline__ void unpack2(uint32_t w, float &lo, float &hi) {
  lo = elem_to_f32<DT>((uint16_t)(w & 0xffffu));
  hi = elem_to_f32<DT>((uint16_t)(w >> 16));
}
// two binary32 values -> two 16-bit patterns, round to nearest even
template <int DT> __device__ __forceinline__ uint32_t pack_round2(float a, float b);
template <> __device__ __forceinline__ uint32_t pack_round2<0>(float a, float b) {
  typedef _Float16 h2 __attribute__((ext_vector_type(2)));
  typedef float f2 __attribute__((ext_vector_type(2)));
  const f2 v = {a, b};
  return __builtin_bit_cast(uint32_t, __builtin_convertvector(v, h2));
}
template <> __device__ __forceinline__ uint32_t pack_round2<1>(float a, float b) {
  typedef __bf16 bf2 __attribute__((ext_vector_type(2)));
  typedef float f2 __attribute__((ext_vector_type(2)));
  const f2 v = {a, b};
  return __builtin_bit_cast(uint32_t, __builtin_convertvector(v, bf2));   // v_cvt_pk_bf16_f32
}
// (int)y truncated toward zero, its low 8 bits written to byte B of acc: one instruction per element (the conversion's
// sub-dword destination select) instead of a conversion plus shifts and ors.  Byte 0 clears the other three bytes, bytes
// 1-3 keep them, so four calls in ascending order build a packed word without an initial value.
template <int B>
__device__ __forceinline__ void cvt_trunc_to_byte(uint32_t &acc, float y) {
  if constexpr (B == 0) asm("v_cvt_i32_f32_sdwa %0, %1 dst_sel:BYTE_0 dst_unused:UNUSED_PAD src0_sel:DWORD" : "=v"(acc) : "v"(y));
  else if constexpr (B == 1) asm("v_cvt_i32_f32_sdwa %0, %1 dst_sel:BYTE_1 dst_unused:UNUSED_PRESERVE src0_sel:DWORD" : "+v"(acc) : "v"(y));
  else if constexpr (B == 2) asm("v_cvt_i32_f32_sdwa %0, %1 dst_sel:BYTE_2 dst_unused:UNUSED_PRESERVE src0_sel:DWORD" : "+v"(acc) : "v"(y));
  else asm("v_cvt_i32_f32_sdwa %0, %1 dst_sel:BYTE_3 dst_unused:UNUSED_PRESERVE src0_sel:DWORD" : "+v"(acc) : "v"(y));
}
// Hides a register's value from the optimiser: placed between two passes over the packed tile, it keeps the compiler
// from carrying the widened (binary32) copies of one pass over to the next, which would double the registers again.
__device__ __forceinline__ void forget(uint32_t &v) { asm volatile("" : "+v"(v)); }
__device__ __forceinline__ uint32_t wave_max_u32(uint32_t v) {
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) v = max(v, (uint32_t)__shfl_xor((int)v, o, SPG_WAVE));
  return v;
}

// Sums of eight columns over the four 16-lane rows of a wavefront (bits 4 and 5 of the lane): half the columns change places
// with the other half's lanes, the two add up, and again.  Lane l ends with columns 4 * bit 5 + 2 * bit 4 + {0, 1}: a quarter
// of the LDS space and of its writes and reads for the rest of the column sum.  (With the full set in LDS, 32 KiB held a CU
// to four workgroups of the back kernel: 30 heads N17776 D64 55.8 us, with 10 KiB and word-wide V tile writes 44.0 us.)
template <int M>
__device__ __forceinline__ double swap_add_f64(double a, double b) {
  const uint64_t ua = __builtin_bit_cast(uint64_t, a), ub = __builtin_bit_cast(uint64_t, b);
  uint32_t al = (uint32_t)ua, ah = (uint32_t)(ua >> 32), bl = (uint32_t)ub, bh = (uint32_t)(ub >> 32);
  if constexpr (M == 32) asm volatile("s_nop 1\n\tv_permlane32_swap_b32 %0, %1\n\tv_permlane32_swap_b32 %2, %3" : "+v"(al), "+v"(bl), "+v"(ah), "+v"(bh));
  else asm volatile("s_nop 1\n\tv_permlane16_swap_b32 %0, %1\n\tv_permlane16_swap_b32 %2, %3" : "+v"(al), "+v"(bl), "+v"(ah), "+v"(bh));
  return __builtin_bit_cast(double, ((uint64_t)ah << 32) | al) + __builtin_bit_cast(double, ((uint64_t)bh << 32) | bl);
}
__device__ __forceinline__ double2 fold_columns(const double (&x)[8]) {
  double y[4];
#pragma unroll
  for (int i = 0; i < 4; i++) y[i] = swap_add_f64<32>(x[i], x[i + 4]);
  return make_double2(swap_add_f64<16>(y[0], y[2]), swap_add_f64<16>(y[1], y[3]));
}

// One workgroup handles ROWS consecutive rows of one (batch, head), by default 128: one 128-row block or two 64-row blocks (SUB), so
// that the per-block tail (column reduction, pooled mean, flag, scale) is spread over all four wavefronts in both cases.
// QR = rows that share one INT8 scale: BS (per-block granularity, what the reference's operators use) or 32 rows of a
// 128-row Q block (per-warp granularity: quant_per_block.py:102-148 with WARPQ = 32, one scale per 32 query rows, which
// are the rows of one wavefront of the attention kernel).  Pooling and the similarity flag stay per block.
// MEAN: 0 no mean (Q), 1 the finished column mean `km`, 2 the partial column sums km_part (km_chunks per head) that
// km_partial_body wrote - every workgroup adds them up for itself, which takes the small kernel in between out of the
// launch chain and pays while there are few chunks - 3 nothing but x: every workgroup sums the columns of its whole head.
enum { MEAN_NONE = 0, MEAN_GIVEN = 1, MEAN_PARTIAL = 2, MEAN_HERE = 3 };
// NT threads work on ROWS rows: 256 on 128 where there are enough workgroups to fill the chip, more threads on fewer rows
// where there are not and the time is the length of one thread's work.
template <int BS, int D, int NT = 256, int ROWS = 128> constexpr int psq_lds() { return ROWS / BS * (NT / 64 * 128 / D) * D * 8; }
// Where the results go: device memory as the stages hand it on (PsqStore), or the attention kernel's LDS (attn.hip).
// ALL_ROWS: rows beyond the end are written, too (as zeros).  one_scale(): the groups of QR rows
// share the scale of their block after all, so that one instantiation serves both granularities.
template <int D>
struct PsqStore {
  static constexpr bool ALL_ROWS = false;
  uint16_t *pool_at;                  // of the workgroup's first block, row and group
  uint8_t *sim_at;
  int8_t *xq_at;
  float *scale_at;
  __device__ __forceinline__ bool one_scale() const { return false; }
  __device__ __forceinline__ void pool(int sb, int col, uint16_t v) const { pool_at[sb * D + col] = v; }
  __device__ __forceinline__ void sim(int sb, bool v) const { sim_at[sb] = v ? 1 : 0; }
  __device__ __forceinline__ void codes(int row, int c, uint2 v) const { *(uint2 *)(xq_at + (size_t)row * D + c * 8) = v; }
  __device__ __forceinline__ void scale(int g, float v) const { scale_at[g] = v; }
};

// xh: first row of the (batch, head), sn: elements from row to row, wg: number of the ROWS rows; NT: threads of the workgroup
template <int BS, int D, int DT, int MEAN, bool WITH_POOL, int QR, int NT, int ROWS, class Out>
__device__ __forceinline__ void psq_core(const uint16_t *__restrict__ xh, long long sn, const uint16_t *__restrict__ km,
                                         const double *__restrict__ km_part, int km_chunks, const float simthr, int N, int wg, int bh,
                                         unsigned char *smem, const Out &out) {
#pragma clang fp contract(off)
  constexpr int SUB = ROWS / BS;      // blocks per workgroup
  constexpr int TPR = D / 8;          // lanes per row (16 B each)
  constexpr int RPP = NT / TPR;       // rows per pass of the workgroup
  constexpr int NWV = NT / 64;        // wavefronts
  constexpr int NPT = ROWS / RPP;     // passes (rows per thread)
  constexpr int NP = BS / RPP;        // passes per block
  constexpr int WPS = D / 64;         // wavefronts that hold one block's columns in the tail (thread = block * D + column)
  constexpr int NQG = ROWS / QR;      // quantisation groups per workgroup (1, 2 or 4)
  constexpr int GPB = BS / QR;        // ... per block
  constexpr int NPQ = QR / RPP;       // passes per quantisation group
  static_assert(BS == 64 || BS == 128, "block sizes of the operators");
  static_assert(QR == BS || (QR == 32 && BS == 128), "per-block, or 32-row groups of a Q block");
  static_assert(RPP <= QR, "a pass of the workgroup stays inside one quantisation group");
  static_assert(RPP <= BS && SUB >= 1 && SUB * D <= NT, "thread <-> (block, column) mapping of the tail");
  // magnitude patterns (sign bit cleared) order like the magnitudes, for both 16-bit formats
  constexpr uint32_t ABS2 = 0x7fff7fffu;
  constexpr uint32_t INF16 = DT == 1 ? 0x7f80u : 0x7c00u;
  // "every element of the row is tiny": bfloat16 below 2^-63 (both top exponent bits clear), binary16 zero
  constexpr uint32_t TINY2 = DT == 1 ? 0x60006000u : 0x7fff7fffu;
  constexpr bool HAS_MEAN = MEAN != MEAN_NONE;
  const int tid = threadIdx.x, c = tid % TPR, r = tid / TPR;
  const int row_base = wg * ROWS;
  const int rows_here = min(ROWS, N - row_base);          // >= 1
  const bool partial = rows_here < ROWS;                  // workgroup-uniform: only the last workgroup of a head
  auto rows_valid_of = [&](int sb) { return max(0, min(BS, rows_here - sb * BS)); };
  const uint16_t *xb = xh + (size_t)row_base * sn + c * 8;

  // all loads of the thread are issued before the first use (rows beyond the end re-read the last row and are zeroed
  // afterwards: no load sits behind a branch)
  uint32_t w[NPT][4];
  {
    uint4 raw[NPT];
#pragma unroll
    for (int p = 0; p < NPT; p++) raw[p] = load_stream_u4(xb + (size_t)min(r + p * RPP, rows_here - 1) * sn);
#pragma unroll
    for (int p = 0; p < NPT; p++) { w[p][0] = raw[p].x; w[p][1] = raw[p].y; w[p][2] = raw[p].z; w[p][3] = raw[p].w; }
  }
  if constexpr (HAS_MEAN) {
    float kmf[8];
    uint4 v;
    if constexpr (MEAN == MEAN_GIVEN) {
      v = *(const uint4 *)(km + (size_t)bh * D + c * 8);
    } else if constexpr (MEAN == MEAN_HERE) {
      // (the sums are exact in binary64: their order is free)
      constexpr int SG = NWV * 128 / D;                // partial sums per column (fold_columns)
      double(*s_part)[D] = (double(*)[D])smem;
      uint16_t *s_km = (uint16_t *)(smem + SG * D * 8);
      const uint16_t *hb = xh + c * 8;
      double acc[8];
#pragma unroll
      for (int e = 0; e < 8; e++) acc[e] = 0.0;
#pragma unroll 8
      for (int row = r; row < N; row += RPP) {
        const uint4 q = *(const uint4 *)(hb + (size_t)row * sn);
        const uint32_t qw[4] = {q.x, q.y, q.z, q.w};
#pragma unroll
        for (int j = 0; j < 4; j++) {
          float f0, f1;
          unpack2<DT>(qw[j], f0, f1);
          acc[2 * j] += (double)f0;
          acc[2 * j + 1] += (double)f1;
        }
      }
      const int sg = D == 128 ? tid >> 6 : tid >> 6 << 1 | (tid >> 3 & 1);
      *(double2 *)&s_part[sg][c * 8 + (tid >> 5 & 1) * 4 + (tid >> 4 & 1) * 2] = fold_columns(acc);
      __syncthreads();
      if (tid < D) {
        double t = 0.0;
#pragma unroll
        for (int u = 0; u < SG; u++) t += s_part[u][tid];
        s_km[tid] = f64_to_elem<DT>(t / (double)N);
      }
      __syncthreads();
      v = *(const uint4 *)(s_km + c * 8);
      __syncthreads();                                // the LDS is used again below
    } else {
      // (the sums are exact in binary64: their order is free)
      constexpr int G = NT / D;
      double *s_sub = (double *)smem;
      uint16_t *s_km = (uint16_t *)(smem + NT * 8);
      double s = 0.0;
#pragma unroll 4
      for (int i = tid / D; i < km_chunks; i += G) s += km_part[((size_t)bh * km_chunks + i) * D + tid % D];
      s_sub[tid] = s;
      __syncthreads();
      if (tid < D) {
        double t = s_sub[tid];
#pragma unroll
        for (int u = 1; u < G; u++) t += s_sub[tid + u * D];
        s_km[tid] = f64_to_elem<DT>(t / (double)N);
      }
      __syncthreads();
      v = *(const uint4 *)(s_km + c * 8);
      __syncthreads();                                // the LDS is used again below
    }
    unpack2<DT>(v.x, kmf[0], kmf[1]);
    unpack2<DT>(v.y, kmf[2], kmf[3]);
    unpack2<DT>(v.z, kmf[4], kmf[5]);
    unpack2<DT>(v.w, kmf[6], kmf[7]);
    // (k - km) rounded once to the input dtype (utils.py:184-188).  The binary32 difference of two 16-bit floats is
    // either exact or nowhere near a rounding tie of the 16-bit format, so rounding it to nearest even equals rounding
    // the exact difference.  The tile is kept as the rounded 16-bit patterns.
#pragma unroll
    for (int p = 0; p < NPT; p++)
#pragma unroll
      for (int j = 0; j < 4; j++) {
        float f0, f1;
        unpack2<DT>(w[p][j], f0, f1);
        w[p][j] = pack_round2<DT>(f0 - kmf[2 * j], f1 - kmf[2 * j + 1]);
      }
  }
  if (partial) {                                  // masked rows are zero (utils.py:188)
#pragma unroll
    for (int p = 0; p < NPT; p++)
      if (r + p * RPP >= rows_here) { w[p][0] = 0; w[p][1] = 0; w[p][2] = 0; w[p][3] = 0; }
  }

  // largest magnitude of the thread's elements per quantisation group (as 16-bit patterns: group g in half g % 2 of
  // word g / 2) and, per row, whether all of the thread's elements are tiny
  constexpr int MW = (NQG + 1) / 2;
  uint32_t m_thread[MW], tiny_rows = 0;
#pragma unroll
  for (int i = 0; i < MW; i++) m_thread[i] = 0;
#pragma unroll
  for (int g = 0; g < NQG; g++) {
    uint32_t m2 = 0;
#pragma unroll
    for (int p = g * NPQ; p < (g + 1) * NPQ; p++) {
      const uint32_t rm = pk_max_u16(pk_max_u16(w[p][0] & ABS2, w[p][1] & ABS2), pk_max_u16(w[p][2] & ABS2, w[p][3] & ABS2));
      m2 = pk_max_u16(m2, rm);
      if constexpr (WITH_POOL) tiny_rows |= ((rm & TINY2) == 0 ? 1u : 0u) << p;
    }
    m_thread[g / 2] |= max(m2 & 0xffffu, m2 >> 16) << (16 * (g % 2));
  }
  // A NaN pattern lies above the infinity pattern and wins the maxima above.  The similarity flag wants exactly that
  // (a block with a NaN is never "similar"), the quantisation scale does not: the reference's block maximum ignores NaN
  // (tl.max lowers to a maxnum, utils.py:140 / 206), so only the NaN elements themselves are poisoned (they quantise to
  // 0).  m_raw keeps the maxima with NaN for the flag; a thread that met one recomputes m_thread without (rare).
  uint32_t m_raw[MW];
#pragma unroll
  for (int i = 0; i < MW; i++) m_raw[i] = m_thread[i];
  {
    bool nan_seen = false;
#pragma unroll
    for (int i = 0; i < MW; i++) nan_seen |= (m_thread[i] & 0xffffu) > INF16 || (m_thread[i] >> 16) > INF16;
    if (nan_seen) {
#pragma unroll
      for (int i = 0; i < MW; i++) m_thread[i] = 0;
#pragma unroll
      for (int g = 0; g < NQG; g++) {
        uint32_t m1 = 0;
#pragma unroll
        for (int p = g * NPQ; p < (g + 1) * NPQ; p++)
#pragma unroll
          for (int j = 0; j < 4; j++) {
            const uint32_t lo = w[p][j] & 0x7fffu, hi = (w[p][j] >> 16) & 0x7fffu;
            m1 = max(m1, max(lo > INF16 ? 0u : lo, hi > INF16 ? 0u : hi));
          }
        m_thread[g / 2] |= m1 << (16 * (g % 2));
      }
    }
  }
  // largest magnitude pattern of block sb as this thread (or, after the reduction, the workgroup) knows it
  auto block_max = [&](const uint32_t(&mm)[MW], int sb) -> uint32_t {
    uint32_t m = 0;
#pragma unroll
    for (int g = sb * GPB; g < (sb + 1) * GPB; g++) m = max(m, (mm[g / 2] >> (16 * (g % 2))) & 0xffffu);
    return m;
  };
  __shared__ uint32_t s_wmax[NWV][MW], s_wbad[NWV];
  __shared__ long long s_wg[NWV];
#pragma unroll
  for (int i = 0; i < MW; i++) {
    uint32_t mw = m_thread[i];                    // two groups' maxima reduced together
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) mw = pk_max_u16(mw, (uint32_t)__shfl_xor((int)mw, o, SPG_WAVE));
    if ((tid & 63) == 0) s_wmax[tid >> 6][i] = mw;
  }

  if constexpr (WITH_POOL) {
    // column sums of all blocks of the workgroup, one line per wavefront (two at D = 64: fold_columns); used for the pooled mean first and, with a
    // non-negative similarity threshold, for the normalised rows afterwards
    constexpr int RG = NWV * 128 / D;
    double(*s_red)[RG][D] = (double(*)[RG][D])smem;
    const int rg = D == 128 ? tid >> 6 : tid >> 6 << 1 | (tid >> 3 & 1);
    const int rg_col = c * 8 + (tid >> 5 & 1) * 4 + (tid >> 4 & 1) * 2;
    // column sums for the pooled mean: binary64, exact
#pragma unroll
    for (int sb = 0; sb < SUB; sb++) {
      double colsum[8];
#pragma unroll
      for (int e = 0; e < 8; e++) colsum[e] = 0.0;
#pragma unroll
      for (int p = sb * NP; p < (sb + 1) * NP; p++)
#pragma unroll
        for (int j = 0; j < 4; j++) {
          float f0, f1;
          forget(w[p][j]);
          unpack2<DT>(w[p][j], f0, f1);
          colsum[2 * j] += (double)f0;
          colsum[2 * j + 1] += (double)f1;
        }
      *(double2 *)&s_red[sb][rg][rg_col] = fold_columns(colsum);
    }

    // row norms: the TPR lanes of a row group all need sqrt(sum of squares) and its reciprocal for each of their NPT
    // rows.  Both are computed ONCE per NPT rows - lane c of the group takes row c % NPT - and handed round with lane
    // reads, instead of NPT times in every lane.
    static_assert(NPT <= TPR, "one lane of the row group per row");
    // A NEGATIVE similarity threshold (the top-k operators' default, -0.1) decides the flag without the normalised rows:
    // the statistic is ||sum of x_hat||^2 / rows^2 >= 0 > threshold whenever every x_hat is finite.  x_hat = x / norm is
    // non-finite exactly for rows with norm == 0 (all-zero rows such as the padding of a partial block, or rows too
    // small for their squares) and for non-finite x; |x| <= norm (1 + 2^-23) keeps every other quotient within fp16.
    // Only two facts about the rows are needed then: is any element non-finite, and does any row have a zero norm.  A
    // row whose largest |x| is at least 2^-63 has a sum of squares of at least 2^-126, a positive binary32 number; rows
    // in which every element is smaller (all-zero rows, the padding of a partial block, bfloat16 values near the bottom
    // of the range) are decided by the exact sums below.
    const bool sim_trivial = simthr < 0.f;     // workgroup-uniform
    uint32_t bad = 0;                                  // bit sb: block sb holds a non-finite x_hat
    float ssf_mine = 0.f;
    bool need_norms = true;                            // wavefront-uniform
    if (sim_trivial) {
#pragma unroll
      for (int sb = 0; sb < SUB; sb++)                 // inf or NaN anywhere (overflowing squares of finite values are harmless: x / inf = 0)
        bad |= (block_max(m_raw, sb) >= INF16 ? 1u : 0u) << sb;
      tiny_rows = group_and_u32<TPR>(tiny_rows);      // rows tiny in every lane of their group
      need_norms = __any(tiny_rows != 0);             // rare
    }
    if (need_norms) {
      // sum of squares of every row (exact in binary64), rounded to binary32 like the reference's (utils.py:194)
#pragma unroll
      for (int p = 0; p < NPT; p++) {
        double ss = 0.0;
#pragma unroll
        for (int j = 0; j < 4; j++) {
          float f0, f1;
          forget(w[p][j]);
          unpack2<DT>(w[p][j], f0, f1);
          const double d0 = (double)f0, d1 = (double)f1;
          ss = __builtin_fma(d0, d0, ss);             // squares and their sum are exact in binary64
          ss = __builtin_fma(d1, d1, ss);
        }
        ss = group_sum_f64<TPR>(ss);                 // the TPR lanes of this row
        const float ssf = (float)ss;
        ssf_mine = (c % NPT == p) ? ssf : ssf_mine;
        if (sim_trivial) bad |= ((ssf == 0.f) ? 1u : 0u) << (p / NP);
      }
    }
    __syncthreads();
    // tail: thread = block * D + column
    const int t_sb = tid / D, t_col = tid % D;
    const bool t_on = tid < SUB * D;
    const int t_rows = rows_valid_of(t_sb);
    if (t_on && t_rows > 0) {
      double s = 0.0;
      #pragma unroll
      for (int i = 0; i < RG; i++) s += s_red[t_sb][i][t_col];
      // full blocks: the row count is a power of two, so the product with its reciprocal is the exact quotient
      const double mean = t_rows == BS ? s * (1.0 / BS) : s / (double)t_rows;
      out.pool(t_sb, t_col, f64_to_elem_fast<DT>(mean));
    }
    long long g = 0;
    if (!sim_trivial) {
      __syncthreads();                                // s_red is reused
      const float norm_mine = sqrtf(ssf_mine);
      const float rn_mine = rcp_safe(norm_mine) ? exact_rcp(norm_mine) : 0.f;
      const int group_lane0 = (tid & 63) & ~(TPR - 1);
#pragma unroll
      for (int sb = 0; sb < SUB; sb++) {
        double colxh[8];
#pragma unroll
        for (int e = 0; e < 8; e++) colxh[e] = 0.0;
#pragma unroll
        for (int p = sb * NP; p < (sb + 1) * NP; p++) {
          const float norm = __shfl(norm_mine, group_lane0 + p, SPG_WAVE);
          const float rn = __shfl(rn_mine, group_lane0 + p, SPG_WAVE);
          const bool fast = rcp_safe(norm);
#pragma unroll
          for (int j = 0; j < 4; j++) {
            float f0, f1;
            forget(w[p][j]);
            unpack2<DT>(w[p][j], f0, f1);
            // the slow branch gives 0/0 = NaN for all-zero (masked) rows
            const _Float16 h0 = (_Float16)(fast ? div_by(f0, norm, rn) : f0 / norm);
            const _Float16 h1 = (_Float16)(fast ? div_by(f1, norm, rn) : f1 / norm);
            colxh[2 * j] += (double)(float)h0;        // fp16 values: integer multiples of 2^-24, sums are exact
            colxh[2 * j + 1] += (double)(float)h1;
          }
        }
        *(double2 *)&s_red[sb][rg][rg_col] = fold_columns(colxh);
      }
      __syncthreads();
      if (t_on) {
        double sx = 0.0;
        #pragma unroll
        for (int i = 0; i < RG; i++) sx += s_red[t_sb][i][t_col];
        if (__builtin_isfinite(sx)) {
          const long long si = (long long)(sx * 16777216.0);   // exact integer
          g = si * si;
        } else {
          bad |= 1u << t_sb;                          // a NaN/inf x_hat anywhere in the column
        }
      }
#pragma unroll
      for (int o = 32; o >= 1; o >>= 1) g += shfl_xor_i64(g, o);
      if ((tid & 63) == 0) s_wg[tid >> 6] = g;
    }
    // bit sb of any_bad: some thread saw a non-finite x_hat in block sb (one flag word per wavefront, combined below)
    {
      uint32_t wb = 0;
#pragma unroll
      for (int sb = 0; sb < SUB; sb++) wb |= (__any((bad >> sb) & 1u) ? 1u : 0u) << sb;
      if ((tid & 63) == 0) s_wbad[tid >> 6] = wb;
    }
    __syncthreads();
    uint32_t any_bad = 0;
#pragma unroll
    for (int i = 0; i < NWV; i++) any_bad |= s_wbad[i];
    if (tid < SUB && rows_valid_of(tid) > 0) {
      const int rv = rows_valid_of(tid);
      bool similar = sim_trivial;
      if (!sim_trivial) {
        long long gt = 0;                             // = sum(gram) * 2^48, exact
        for (int i = 0; i < WPS; i++) gt += s_wg[tid * WPS + i];
        const double thr = (double)simthr * (double)(rv * rv) * 281474976710656.0;
        similar = (double)gt > thr;
      }
      out.sim(tid, !((any_bad >> tid) & 1u) && similar);
    }
  } else {
    __syncthreads();
  }

  uint32_t m_all[MW];
#pragma unroll
  for (int i = 0; i < MW; i++) {
    m_all[i] = s_wmax[0][i];
#pragma unroll
    for (int wv = 1; wv < NWV; wv++) m_all[i] = pk_max_u16(m_all[i], s_wmax[wv][i]);
  }
  if (NQG > 1 && out.one_scale()) {
    static_assert(NQG <= 4, "two words of maxima");
    uint32_t m = m_all[0];
    if constexpr (MW == 2) m = pk_max_u16(m, m_all[1]);
    m = max(m & 0xffffu, m >> 16);
#pragma unroll
    for (int i = 0; i < MW; i++) m_all[i] = m | (m << 16);
  }
  // The scale of group g, its reciprocal and the multiplier of its codes.  With four groups a wavefront works out one of them for the whole
  // workgroup: the test takes it as long as the codes of a group's rows (per-warp scales, H47 N384 D64 CDF with FP16 PV 28.5 / 28.0 us per call, H43 N299 D128 27.3 / 26.8, H30 N3000 D128 fp16 97.4 / 96.5).
  auto scale_of = [&](int g) {
    const float amax = elem_to_f32<DT>((uint16_t)(m_all[g / 2] >> (16 * (g % 2))));
    return amax / 127.0f + 1e-7f;
  };
  auto multiplier = [](float s, float rs) { return rcp_safe(s) ? code_multiplier<DT>(s, rs) : 0.f; };
  __shared__ float s_code[NQG == 4 ? 4 : 1][3];
  const bool shared_test = NQG == 4 && !out.one_scale();
  if (shared_test) {
    const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
    if (wv < 4) {
      float s = scale_of(0);
#pragma unroll
      for (int g = 1; g < NQG; g++) s = wv == g ? scale_of(g) : s;
      const float rs = exact_rcp(s), m = multiplier(s, rs);
      if ((tid & 63) == 0) { s_code[wv % NQG][0] = s; s_code[wv % NQG][1] = rs; s_code[wv % NQG][2] = m; }
    }
    __syncthreads();
  }
  float s, rs, m;
#pragma unroll
  for (int g = 0; g < NQG; g++) {
    // per-block scales exist for blocks with at least one row; the 32-row groups of the last Q block all get a scale
    // (1e-7 for a group without rows, what the reference's quantiser writes for an all-masked group)
    if (QR == BS && rows_here - g * QR <= 0) break;     // workgroup-uniform
    if (shared_test) {
      s = s_code[g][0]; rs = s_code[g][1]; m = s_code[g][2];
    } else if (g == 0 || NQG < 4) {
      s = scale_of(g);
      rs = exact_rcp(s);
      m = multiplier(s, rs);
    }
    auto quantise = [&](auto code4, auto check_rows) {
#pragma unroll
      for (int p = g * NPQ; p < (g + 1) * NPQ; p++) {
        const int row = r + p * RPP;
        if (!decltype(check_rows)::value || Out::ALL_ROWS || row < rows_here) {
          float f[8];
#pragma unroll
          for (int j = 0; j < 4; j++) {
            forget(w[p][j]);
            unpack2<DT>(w[p][j], f[2 * j], f[2 * j + 1]);
          }
          const uint32_t pk0 = code4(f[0], f[1], f[2], f[3]), pk1 = code4(f[4], f[5], f[6], f[7]);
          out.codes(row, c, make_uint2(pk0, pk1));
        }
      }
    };
    auto all_rows = [&](auto code4) {
      if (Out::ALL_ROWS || !partial) quantise(code4, std::false_type{});     // (the common case carries no row test)
      else quantise(code4, std::true_type{});
    };
    // One fma and three quarters of a permute per element where a multiplier gives the codes (a NaN, which the maximum leaves out,
    // passes through the fma with a zero low byte: the low mantissa bits of a widened 16-bit float are zero), otherwise the division:
    // truncation toward zero, low 8 bits of element e into byte e % 4 (a -0 quotient truncates to 0 either way, a NaN, too).
    auto product = [&](float f0, float f1, float f2, float f3) {
      return pack_codes(__builtin_fmaf(f0, m, CODE_MAGIC), __builtin_fmaf(f1, m, CODE_MAGIC), __builtin_fmaf(f2, m, CODE_MAGIC), __builtin_fmaf(f3, m, CODE_MAGIC));
    };
    auto divided = [&](auto divide) {
      return [&, divide](float f0, float f1, float f2, float f3) {
        uint32_t pk;
        cvt_trunc_to_byte<0>(pk, away_from_zero(divide(f0)));
        cvt_trunc_to_byte<1>(pk, away_from_zero(divide(f1)));
        cvt_trunc_to_byte<2>(pk, away_from_zero(divide(f2)));
        cvt_trunc_to_byte<3>(pk, away_from_zero(divide(f3)));
        return pk;
      };
    };
    if (m != 0.f) all_rows(product);                       // workgroup-uniform
    else if (rcp_safe(s)) all_rows(divided([&](float v) { return div_by(v, s, rs); }));
    else quantise(divided([&](float v) { return v / s; }), std::true_type{});
    if (tid == 0) out.scale(g, s);
  }
}
template <int BS, int D, int DT, int MEAN, bool WITH_POOL, int QR = BS, int NT = 256, int ROWS = 128>
__device__ __forceinline__ void psq_body(const uint16_t *__restrict__ x, const Strides &xs,
                                         const uint16_t *__restrict__ km, const double *__restrict__ km_part, int km_chunks,
                                         uint16_t *__restrict__ pool, uint8_t *__restrict__ sim,
                                         int8_t *__restrict__ xq, float *__restrict__ scale,
                                         const float simthr, int H, int N, int nb, int wg, int bh, unsigned char *smem) {
  const size_t blk0 = (size_t)bh * nb + wg * (ROWS / BS);
  PsqStore<D> out;
  out.pool_at = pool + blk0 * D;
  out.sim_at = sim + blk0;
  out.xq_at = xq + ((size_t)bh * N + (size_t)wg * ROWS) * D;
  out.scale_at = scale + blk0 * (BS / QR);
  psq_core<BS, D, DT, MEAN, WITH_POOL, QR, NT, ROWS>(x + (size_t)(bh / H) * xs.sb + (size_t)(bh % H) * xs.sh, xs.sn, km, km_part, km_chunks,
                                                     simthr, N, wg, bh, smem, out);
}

// exclusive prefix of per-thread counts over the NT threads of the workgroup; returns (offset, total)
template <int NT>
__device__ __forceinline__ int2 block_exclusive_scan_i32(int v, int *s_tmp /* >= NT / 64 ints */) {
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  int inc = v;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const int t = __shfl_up(inc, o, SPG_WAVE);
    if (lane >= o) inc += t;
  }
  __syncthreads();                       // s_tmp may still be read from a previous call
  if (lane == 63) s_tmp[wave] = inc;
  __syncthreads();
  int base = 0, total = 0;
#pragma unroll
  for (int w = 0; w < NT / 64; w++) {
    const int t = s_tmp[w];
    if (w < wave) base += t;
    total += t;
  }
  return make_int2(base + inc - v, total);
}

// flags (per column, via functor) -> ascending compact index list -> delta LUT, zero tail, valid count.
template <int NT, class FlagFn>
__device__ __forceinline__ void emit_lut(FlagFn flag, int nk, int nkp, int32_t *s_idx, int *s_tmp,
                                         int32_t *__restrict__ lut_row, int32_t *__restrict__ valid_out) {
  const int tid = threadIdx.x;
  const int seg = nkp / NT;
  const int j0 = tid * seg, j1 = min(nk, j0 + seg);
  int cnt = 0;
  for (int j = j0; j < j1; j++) cnt += flag(j) ? 1 : 0;
  const int2 st = block_exclusive_scan_i32<NT>(cnt, s_tmp);
  int pos = st.x;
  for (int j = j0; j < j1; j++)
    if (flag(j)) s_idx[pos++] = j;
  __syncthreads();
  for (int p = tid; p < nk; p += NT) {
    int v = 0;
    if (p < st.y) v = s_idx[p] - (p ? s_idx[p - 1] : 0);
    lut_row[p] = v;
  }
  if (tid == 0) *valid_out = st.y;
}

// =============================================================================================
// user mask -> LUT
// =============================================================================================
template <int KIND>
__device__ __forceinline__ bool mask_nonzero(const void *row, int j) {
  if constexpr (KIND == 0) return ((const uint8_t *)row)[j] != 0;
  if constexpr (KIND == 1) return ((const uint16_t *)row)[j] != 0;
  if constexpr (KIND == 2) return ((const uint32_t *)row)[j] != 0;
  if constexpr (KIND == 3) return ((const uint64_t *)row)[j] != 0;
  if constexpr (KIND == 4) return (((const uint16_t *)row)[j] & 0x7fffu) != 0;            // +-0.0 is zero
  if constexpr (KIND == 5) return (((const uint32_t *)row)[j] & 0x7fffffffu) != 0;
  if constexpr (KIND == 6) return (((const uint64_t *)row)[j] & 0x7fffffffffffffffull) != 0;
  return false;
}
constexpr int mask_elem_size(int kind) { return kind == 0 ? 1 : (kind == 1 || kind == 4) ? 2 : (kind == 2 || kind == 5) ? 4 : 8; }

// one row of a user mask -> LUT row; LDS: 4 * nkp bytes for the index list, 64 for the scan; nkp is a multiple of NT
template <int KIND, int NT = 256>
__device__ __forceinline__ void map_to_lut_body(const void *__restrict__ mask, int32_t *__restrict__ lut,
                                                int32_t *__restrict__ valid, int nk, int nkp, size_t row_id,
                                                unsigned char *smem) {
  int32_t *s_idx = (int32_t *)(smem + 64);
  const size_t row_off = row_id * nk;
  const void *row = (const unsigned char *)mask + row_off * mask_elem_size(KIND);
  auto flag = [&](int j) -> bool { return mask_nonzero<KIND>(row, j); };
  emit_lut<NT>(flag, nk, nkp, s_idx, (int *)smem, lut + row_off, valid + row_id);
}

// =============================================================================================
// V path
// =============================================================================================
template <int DT>
__device__ __forceinline__ float elem_to_f16_f32(uint16_t b) {
  // value of the element after the cast to fp16 the reference applies to V (core.py:117)
  if constexpr (DT == 0) return elem_to_f32<0>(b);
  const _Float16 h = (_Float16)elem_to_f32<1>(b);
  return (float)h;
}

// Largest |fp16(v)| of every channel over one chunk of rows.  store(d, value) receives the result of channel d.
template <int D, int NT = 256> constexpr int v_absmax_lds() { return NT / (D / 8) * D * 4; }
template <int D, int DT, int NT = 256, class Store>
__device__ __forceinline__ void v_absmax_body(const uint16_t *__restrict__ v, const Strides &vs, int H, int N,
                                              int rows_per_chunk, int chunk, int bh, unsigned char *smem, Store store) {
  constexpr int TPR = D / 8;
  constexpr int RPP = NT / TPR;
  const int c = threadIdx.x % TPR, r = threadIdx.x / TPR;
  const int row0 = chunk * rows_per_chunk;
  const int row1 = min(N, row0 + rows_per_chunk);
  const uint16_t *base = v + (size_t)(bh / H) * vs.sb + (size_t)(bh % H) * vs.sh + c * 8;
  // The cast to fp16 is monotonic in the magnitude, so the largest |fp16(v)| is the cast of the largest |v|: the maximum
  // is taken on the 16-bit magnitude patterns (which order like the magnitudes), two per instruction, and only the
  // result is converted.
  typedef unsigned short u16x2_t __attribute__((ext_vector_type(2)));
  constexpr uint32_t INF16 = DT == 1 ? 0x7f80u : 0x7c00u;
  uint32_t mp[4] = {0, 0, 0, 0};
#pragma unroll 4
  for (int row = row0 + r; row < row1; row += RPP) {
    const uint4 q = load_stream_u4(base + (size_t)row * vs.sn);
    const uint32_t w[4] = {q.x, q.y, q.z, q.w};
#pragma unroll
    for (int j = 0; j < 4; j++)
      mp[j] = __builtin_bit_cast(uint32_t, __builtin_elementwise_max(__builtin_bit_cast(u16x2_t, mp[j]),
                                                                      __builtin_bit_cast(u16x2_t, w[j] & 0x7fff7fffu)));
  }
  // A NaN pattern lies above the infinity pattern and would win the maximum, whereas the reference's fmaxf / fminf
  // (fused.cu:120-123) ignore NaN: only the NaN elements themselves are poisoned, not their channel's scale.  The
  // common case pays one test; a thread that met a NaN goes over its rows again with the NaN patterns taken as zero.
  if (max(max(mp[0] & 0xffffu, mp[0] >> 16), max(mp[1] & 0xffffu, mp[1] >> 16)) > INF16 ||
      max(max(mp[2] & 0xffffu, mp[2] >> 16), max(mp[3] & 0xffffu, mp[3] >> 16)) > INF16) {
    mp[0] = mp[1] = mp[2] = mp[3] = 0;
    for (int row = row0 + r; row < row1; row += RPP) {
      const uint4 q = *(const uint4 *)(base + (size_t)row * vs.sn);
      const uint32_t w[4] = {q.x, q.y, q.z, q.w};
#pragma unroll
      for (int j = 0; j < 4; j++) {
        uint32_t lo = w[j] & 0x7fffu, hi = (w[j] >> 16) & 0x7fffu;
        lo = lo > INF16 ? 0u : lo;
        hi = hi > INF16 ? 0u : hi;
        mp[j] = max(mp[j] & 0xffffu, lo) | (max(mp[j] >> 16, hi) << 16);
      }
    }
  }
  float m[8];
#pragma unroll
  for (int e = 0; e < 8; e++)
    m[e] = elem_to_f16_f32<DT>((uint16_t)((e & 1) ? (mp[e >> 1] >> 16) : (mp[e >> 1] & 0xffffu)));
  float(*sm)[D] = (float(*)[D])smem;
#pragma unroll
  for (int e = 0; e < 8; e++) sm[r][c * 8 + e] = m[e];
  __syncthreads();
  if (threadIdx.x < D) {
    float s = 0.f;
    for (int i = 0; i < RPP; i++) s = fmaxf(s, sm[i][threadIdx.x]);
    store((int)threadIdx.x, s);
  }
}

// One workgroup per 64-key tile.  LDS holds the transposed tile [D][64] bytes.
// amax_of(d): the channel maximum (a whole-head value, from wherever the kernel has it).
template <int D> constexpr int v_quant_lds() { return D * (64 + 4); }
template <int D, int DT, int NT = 256, class Amax>
__device__ __forceinline__ void v_quant_body(const uint16_t *__restrict__ v, const Strides &vs, int H,
                                             uint8_t *__restrict__ v8, int N, int nk, int blk, int bh, unsigned char *smem,
                                             Amax amax_of) {
  constexpr int TPR = D / 8;
  constexpr int RPP = NT / TPR;
  constexpr int NP = 64 / RPP;
  static_assert(NP == 1 || NP == 2 || NP == 4, "rows per thread");
  constexpr int LDW = 64 + 4;  // padded row (bytes) of the transposed tile
  uint8_t *tile = smem;
  const int tid = threadIdx.x;
  const int c = tid % TPR, r = tid / TPR;
  const uint16_t *base = v + (size_t)(bh / H) * vs.sb + (size_t)(bh % H) * vs.sh + (size_t)blk * 64 * vs.sn + c * 8;
  const int last_row = min(63, N - 1 - blk * 64);
  // A thread takes NP neighbouring rows, so that their codes of one channel leave as one LDS word.
  uint4 raw[NP];                     // every load is issued before the first use; rows beyond N re-read the last row
#pragma unroll
  for (int p = 0; p < NP; p++) raw[p] = load_stream_u4(base + (size_t)min(r * NP + p, last_row) * vs.sn);
  float recp[8];
#pragma unroll
  for (int e = 0; e < 8; e++) recp[e] = 2.25f / amax_of(c * 8 + e);
#pragma unroll
  for (int e = 0; e < 8; e++) {
    float x[4];
#pragma unroll
    for (int p = 0; p < 4; p++) {
      x[p] = 0.f;
      if (p < NP) {
        const uint32_t w[4] = {raw[p % NP].x, raw[p % NP].y, raw[p % NP].z, raw[p % NP].w};
        x[p] = elem_to_f16_f32<DT>((uint16_t)((e & 1) ? (w[e >> 1] >> 16) : (w[e >> 1] & 0xffffu))) * recp[e];
        if (r * NP + p > last_row) x[p] = 0.f;                        // rows beyond N are zero
      }
    }
    int pk = __builtin_amdgcn_cvt_pk_fp8_f32(x[0], x[1], 0, false);
    if constexpr (NP == 4) pk = __builtin_amdgcn_cvt_pk_fp8_f32(x[2], x[3], pk, true);
    uint8_t *const dst = tile + (c * 8 + e) * LDW + r * NP;
    if constexpr (NP == 4) *(uint32_t *)dst = (uint32_t)pk;
    else if constexpr (NP == 2) *(uint16_t *)dst = (uint16_t)pk;
    else *dst = (uint8_t)pk;
  }
  __syncthreads();
  uint8_t *out = v8 + ((size_t)bh * nk + blk) * (size_t)(D * 64);
  for (int i = tid; i < D * 4; i += NT) {   // 16-byte pieces: D rows x 4 slots
    const int d = i >> 2, slot = i & 3;
    const int kc = slot ^ ((d >> 2) & 3);      // key chunk stored in this slot
    const uint32_t *src = (const uint32_t *)(tile + d * LDW + kc * 16);
    *(uint4 *)(out + d * 64 + slot * 16) = make_uint4(src[0], src[1], src[2], src[3]);
  }
}

// V -> fp16 -> V^T tiles [nk][D][64] fp16 for the fp16-PV attention variant.  Inside a 128-byte tile row (one channel,
// 64 keys) the eight 8-key chunks are stored at slot = chunk ^ ((d >> 1) & 7) (the LDS swizzle of the attention kernel).
// Keys at or beyond N are zero.  One workgroup per 64-key tile.
template <int D> constexpr int v_tiles_f16_lds() { return D * (64 + 2) * 2; }
template <int D, int DT, int NT = 256>
__device__ __forceinline__ void v_tiles_f16_body(const uint16_t *__restrict__ v, const Strides &vs, int H,
                                                 uint16_t *__restrict__ vt, int N, int nk, int blk, int bh,
                                                 unsigned char *smem) {
  constexpr int TPR = D / 8;
  constexpr int RPP = NT / TPR;
  constexpr int NP = 64 / RPP;
  constexpr int LDW = 64 + 2;  // padded row (halves) of the transposed tile
  uint16_t *tile = (uint16_t *)smem;
  const int tid = threadIdx.x;
  const int c = tid % TPR, r = tid / TPR;
  const uint16_t *base = v + (size_t)(bh / H) * vs.sb + (size_t)(bh % H) * vs.sh + (size_t)blk * 64 * vs.sn + c * 8;
  const int last_row = min(63, N - 1 - blk * 64);
  uint4 raw[NP];
#pragma unroll
  for (int p = 0; p < NP; p++) raw[p] = load_stream_u4(base + (size_t)min(r + p * RPP, last_row) * vs.sn);
#pragma unroll
  for (int p = 0; p < NP; p++) {
    const int row = r + p * RPP;
    const uint4 q = row <= last_row ? raw[p] : make_uint4(0, 0, 0, 0);
    const uint32_t w[4] = {q.x, q.y, q.z, q.w};
#pragma unroll
    for (int e = 0; e < 8; e++) {
      const uint16_t b = (uint16_t)((e & 1) ? (w[e >> 1] >> 16) : (w[e >> 1] & 0xffffu));
      uint16_t h = b;
      if constexpr (DT == 1) h = f32_to_elem<0>(elem_to_f32<1>(b));     // bf16 -> fp16, one rounding
      tile[(c * 8 + e) * LDW + row] = h;
    }
  }
  __syncthreads();
  uint16_t *out = vt + ((size_t)bh * nk + blk) * (size_t)(D * 64);
  for (int i = tid; i < D * 8; i += NT) {   // 16-byte pieces: D rows x 8 slots
    const int d = i >> 3, slot = i & 7;
    const int kc = slot ^ ((d >> 1) & 7);      // key chunk stored in this slot
    const uint16_t *src = tile + d * LDW + kc * 8;
    uint32_t o[4];
#pragma unroll
    for (int e = 0; e < 4; e++) o[e] = (uint32_t)src[2 * e] | ((uint32_t)src[2 * e + 1] << 16);
    *(uint4 *)(out + d * 64 + slot * 8) = make_uint4(o[0], o[1], o[2], o[3]);
  }
}

}  // namespace spg
