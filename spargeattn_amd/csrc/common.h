// Shared device helpers for the gfx950 SpargeAttn kernels: element conversions with a single rounding,
// wavefront (64-lane) and workgroup reductions, error plumbing for the C ABI.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#define SPG_WAVE 64

namespace spg {

// ---------------------------------------------------------------------------------------------
// 16-bit element types.  DT = 0: IEEE binary16, DT = 1: bfloat16 (same numbering as enum spg_dtype).
// ---------------------------------------------------------------------------------------------
template <int DT> __device__ __forceinline__ float elem_to_f32(uint16_t b);
template <> __device__ __forceinline__ float elem_to_f32<0>(uint16_t b) {
  _Float16 h = __builtin_bit_cast(_Float16, b);
  return (float)h;
}
template <> __device__ __forceinline__ float elem_to_f32<1>(uint16_t b) {
  return __builtin_bit_cast(float, (uint32_t)b << 16);
}

// binary64 -> 16-bit pattern with ONE round-to-nearest-even (never through binary32).
// MANT mantissa bits, BIAS exponent bias, EMIN exponent of the smallest normal.
template <int MANT, int BIAS, int EMIN>
__device__ __forceinline__ uint16_t f64_to_bits16(double x) {
  const uint64_t b = __builtin_bit_cast(uint64_t, x);
  const uint16_t sign = (uint16_t)((b >> 63) << 15);
  const uint64_t a = b & 0x7fffffffffffffffull;
  const double ax = __builtin_bit_cast(double, a);
  constexpr int EXPBITS = 15 - MANT;
  constexpr uint16_t INF = (uint16_t)(((1u << EXPBITS) - 1u) << MANT);
  if (a > 0x7ff0000000000000ull) return sign | INF | (uint16_t)(1u << (MANT - 1));  // NaN
  // largest finite = (2 - 2^-MANT) * 2^(INFEXP-1-BIAS); halfway to the next binade rounds to inf
  constexpr int EMAX = ((1 << EXPBITS) - 2) - BIAS;
  const double ovf = __builtin_ldexp(2.0 - __builtin_ldexp(1.0, -MANT - 1), EMAX);
  if (ax >= ovf) return sign | INF;
  if (ax < __builtin_ldexp(1.0, EMIN)) {
    const double y = __builtin_rint(ax * __builtin_ldexp(1.0, MANT - EMIN));  // count of subnormal quanta
    return sign | (uint16_t)(int)y;
  }
  constexpr int SH = 52 - MANT;
  const uint64_t lsb = (a >> SH) & 1ull;
  const uint64_t r = (a + ((1ull << (SH - 1)) - 1ull) + lsb) >> SH;            // [exp11 | mant]
  return sign | (uint16_t)(r - ((uint64_t)(1023 - BIAS) << MANT));
}

template <int DT> __device__ __forceinline__ uint16_t f64_to_elem(double x);
template <> __device__ __forceinline__ uint16_t f64_to_elem<0>(double x) { return f64_to_bits16<10, 15, -14>(x); }
template <> __device__ __forceinline__ uint16_t f64_to_elem<1>(double x) { return f64_to_bits16<7, 127, -126>(x); }

// binary32 -> 16-bit pattern, RNE (used for outputs that are produced in fp32)
template <int DT> __device__ __forceinline__ uint16_t f32_to_elem(float x);
template <> __device__ __forceinline__ uint16_t f32_to_elem<0>(float x) {
  _Float16 h = (_Float16)x;
  return __builtin_bit_cast(uint16_t, h);
}
template <> __device__ __forceinline__ uint16_t f32_to_elem<1>(float x) {
  return __builtin_bit_cast(uint16_t, (__bf16)x);   // v_cvt_pk_bf16_f32: round to nearest even in hardware
}

// binary64 -> 16-bit pattern (round to nearest even) through binary32 where that provably gives the same bits: the
// first rounding (to 24 bits) can only change the second one when it lands exactly on a rounding tie of the 16-bit
// format, so every other value inside the format's normal range takes two hardware conversions instead of the 64-bit
// integer arithmetic of f64_to_elem; ties, zero-range, subnormal and overflowing values go the exact way.
template <int DT>
__device__ __forceinline__ uint16_t f64_to_elem_fast(double x) {
  const float r = (float)x;                                        // v_cvt_f32_f64
  const uint32_t b = __builtin_bit_cast(uint32_t, r);
  const uint32_t mag = b & 0x7fffffffu;
  constexpr uint32_t DROP = DT == 1 ? 16u : 13u;                   // binary32 mantissa bits the 16-bit format drops
  constexpr uint32_t LOW = (1u << DROP) - 1u, TIE = 1u << (DROP - 1u);
  constexpr uint32_t LO = DT == 1 ? 0x00800000u : 0x38800000u;     // 2^-126 / 2^-14: smallest normal of the format
  constexpr uint32_t HI = DT == 1 ? 0x7f000000u : 0x47000000u;     // 2^127 / 2^15: well below the overflow threshold
  const bool safe = mag == 0u || (mag >= LO && mag < HI && (b & LOW) != TIE);
  return safe ? f32_to_elem<DT>(r) : f64_to_elem<DT>(x);
}

// Round two binary32 values to the 16-bit element type and widen them again (one packed conversion for bfloat16).
template <int DT> __device__ __forceinline__ void round2_through_elem(float &a, float &b);
template <> __device__ __forceinline__ void round2_through_elem<0>(float &a, float &b) {
  a = (float)(_Float16)a;
  b = (float)(_Float16)b;
}
template <> __device__ __forceinline__ void round2_through_elem<1>(float &a, float &b) {
  typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
  typedef float f32x2 __attribute__((ext_vector_type(2)));
  const f32x2 v = {a, b};
  const uint32_t u = __builtin_bit_cast(uint32_t, __builtin_convertvector(v, bf16x2));
  a = __builtin_bit_cast(float, u << 16);
  b = __builtin_bit_cast(float, u & 0xffff0000u);
}

// 16-byte global load with the non-temporal hint: for tensors a kernel streams through once.  On this machine a
// read-only stream reaches 6.6 TB/s with the hint against 5.9 TB/s without.
__device__ __forceinline__ uint4 load_stream_u4(const void *p) {
  typedef unsigned int u4_t __attribute__((ext_vector_type(4)));
  const u4_t t = __builtin_nontemporal_load((const u4_t *)p);
  return make_uint4(t[0], t[1], t[2], t[3]);
}

// ---------------------------------------------------------------------------------------------
// wavefront shuffles for 64-bit values
// ---------------------------------------------------------------------------------------------
__device__ __forceinline__ long long shfl_xor_i64(long long v, int mask) {
  uint64_t u = (uint64_t)v;
  uint32_t lo = (uint32_t)u, hi = (uint32_t)(u >> 32);
  lo = __shfl_xor(lo, mask, SPG_WAVE);
  hi = __shfl_xor(hi, mask, SPG_WAVE);
  return (long long)(((uint64_t)hi << 32) | lo);
}

// Combine the value of lane l with that of lane l^32 (the two 32-lane halves) with one v_permlane32_swap:
// the instruction exchanges lanes 32..63 of its first register with lanes 0..31 of its second, so that afterwards
// the first register holds the lower half's values in both halves and the second the upper half's.
// (Inline asm with two distinct registers: the builtin mis-compiles when both operands are the same value.)
__device__ __forceinline__ void half_swap(float v, float &lo, float &hi) {
  lo = v;
  hi = v;
  asm volatile("s_nop 1\n\tv_permlane32_swap_b32 %0, %1" : "+v"(lo), "+v"(hi));
}
__device__ __forceinline__ float half_swap_max_f32(float v) {
  float lo, hi;
  half_swap(v, lo, hi);
  return fmaxf(lo, hi);
}
__device__ __forceinline__ float half_swap_sum_f32(float v) {
  float lo, hi;
  half_swap(v, lo, hi);
  return lo + hi;
}

// Sum over aligned groups of G lanes (G in {2,4,8,16}) with DPP lane permutes (VALU rate, no LDS traffic).
// Steps: xor 1, xor 2 (quad permutes), then half-row mirror and row mirror, which pair a group with its sibling
// once the values are uniform inside the group.  Every lane of the group ends with the same total.
template <int CTRL>
__device__ __forceinline__ double dpp_f64(double v) {
  const uint64_t u = __builtin_bit_cast(uint64_t, v);
  const int lo = __builtin_amdgcn_update_dpp(0, (int)(uint32_t)u, CTRL, 0xf, 0xf, true);
  const int hi = __builtin_amdgcn_update_dpp(0, (int)(uint32_t)(u >> 32), CTRL, 0xf, 0xf, true);
  return __builtin_bit_cast(double, ((uint64_t)(uint32_t)hi << 32) | (uint32_t)lo);
}
template <int G>
__device__ __forceinline__ double group_sum_f64(double v) {
  if constexpr (G >= 2) v += dpp_f64<0xB1>(v);    // quad_perm [1,0,3,2]
  if constexpr (G >= 4) v += dpp_f64<0x4E>(v);    // quad_perm [2,3,0,1]
  if constexpr (G >= 8) v += dpp_f64<0x141>(v);   // row_half_mirror
  if constexpr (G >= 16) v += dpp_f64<0x140>(v);  // row_mirror
  return v;
}

// Bitwise AND over aligned groups of G lanes (same lane permutes as group_sum_f64).
template <int G>
__device__ __forceinline__ uint32_t group_and_u32(uint32_t v) {
  if constexpr (G >= 2) v &= (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0xB1, 0xf, 0xf, true);
  if constexpr (G >= 4) v &= (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x4E, 0xf, 0xf, true);
  if constexpr (G >= 8) v &= (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x141, 0xf, 0xf, true);
  if constexpr (G >= 16) v &= (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x140, 0xf, 0xf, true);
  return v;
}

// Exchanges over the 64 lanes at VALU rate.  A __shfl_xor is an LDS round trip of 100 clocks and more, and the reductions
// below are chains of six: they stand in the start-up of every row of the attention kernel.
// Lane l receives the value of lane l ^ M.
template <int M>
__device__ __forceinline__ uint32_t lane_xor_u32(uint32_t v) {
  static_assert(M == 1 || M == 2 || M == 4 || M == 8, "inside a row of 16 lanes");
  constexpr int CTRL = M == 1 ? 0xB1 : M == 2 ? 0x4E : M == 4 ? 0x141 : 0x128;   // quad permutes, half-row mirror (l ^ 7), rotate by 8
  const int t = __builtin_amdgcn_update_dpp(0, (int)v, CTRL, 0xf, 0xf, true);
  return (uint32_t)(M == 4 ? __builtin_amdgcn_update_dpp(0, t, 0x1B, 0xf, 0xf, true) : t);        // ... and l ^ 3
}
// a = the value of the lane of the pair (l, l ^ M) whose bit M is clear, b = the other's, in both lanes
template <int M>
__device__ __forceinline__ void pair_of_u32(uint32_t v, uint32_t &a, uint32_t &b) {
  static_assert(M == 16 || M == 32, "rows of 16 lanes");
  a = v;
  b = v;
  if constexpr (M == 32) asm volatile("s_nop 1\n\tv_permlane32_swap_b32 %0, %1" : "+v"(a), "+v"(b));
  else asm volatile("s_nop 1\n\tv_permlane16_swap_b32 %0, %1" : "+v"(a), "+v"(b));
}
template <int M>
__device__ __forceinline__ double pair_sum_f64(double v) {
  const uint64_t u = __builtin_bit_cast(uint64_t, v);
  uint32_t al, bl, ah, bh;
  pair_of_u32<M>((uint32_t)u, al, bl);
  pair_of_u32<M>((uint32_t)(u >> 32), ah, bh);
  return __builtin_bit_cast(double, ((uint64_t)ah << 32) | al) + __builtin_bit_cast(double, ((uint64_t)bh << 32) | bl);
}
// v + (v of lane l ^ 32), then of l ^ 16, 8, 4, 2, 1: the fixed summation tree of the compressed softmax.  (Once the sums agree
// across l ^ 8, a rotation by 4 reaches the value of lane l ^ 4.)
__device__ __forceinline__ double wave_tree_sum_f64(double v) {
  v = pair_sum_f64<32>(v);
  v = pair_sum_f64<16>(v);
  v += dpp_f64<0x128>(v);
  v += dpp_f64<0x124>(v);
  v += dpp_f64<0x4E>(v);
  v += dpp_f64<0xB1>(v);
  return v;
}
__device__ __forceinline__ float wave_max_f32(float v) {
  uint32_t a, b;
  pair_of_u32<32>(__builtin_bit_cast(uint32_t, v), a, b);
  v = fmaxf(__builtin_bit_cast(float, a), __builtin_bit_cast(float, b));
  pair_of_u32<16>(__builtin_bit_cast(uint32_t, v), a, b);
  v = fmaxf(__builtin_bit_cast(float, a), __builtin_bit_cast(float, b));
  v = fmaxf(v, __builtin_bit_cast(float, lane_xor_u32<8>(__builtin_bit_cast(uint32_t, v))));
  v = fmaxf(v, __builtin_bit_cast(float, lane_xor_u32<4>(__builtin_bit_cast(uint32_t, v))));
  v = fmaxf(v, __builtin_bit_cast(float, lane_xor_u32<2>(__builtin_bit_cast(uint32_t, v))));
  v = fmaxf(v, __builtin_bit_cast(float, lane_xor_u32<1>(__builtin_bit_cast(uint32_t, v))));
  return v;
}
__device__ __forceinline__ int wave_sum_i32(int v) {
  uint32_t a, b;
  pair_of_u32<32>((uint32_t)v, a, b);
  pair_of_u32<16>(a + b, a, b);
  uint32_t s = a + b;
  s += lane_xor_u32<8>(s);
  s += lane_xor_u32<4>(s);
  s += lane_xor_u32<2>(s);
  s += lane_xor_u32<1>(s);
  return (int)s;
}

}  // namespace spg
