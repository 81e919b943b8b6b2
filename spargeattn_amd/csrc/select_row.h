// Block selection for one Q block row: the pieces that the selection kernels (maskpred.hip) and the attention kernel's
// in-place selection (attn.hip) share.  The binary64 sequences here are part of the arithmetic contract (maskpred.hip), so
// contraction is switched off where they stand: attn.hip is compiled with it.
#pragma once
#include "common.h"
#include "launch.h"

namespace spg {

// =============================================================================================
// canonical exp: a fixed sequence of binary64 mul / add (no fma), t <= 0.
// =============================================================================================
__device__ __forceinline__ double cexp(double t) {
#pragma clang fp contract(off)
  if (!(t >= -700.0)) return 0.0;
  const double k = __builtin_rint(t * 1.4426950408889634);
  const double r = (t - k * 0.6931471803691238) - k * 1.9082149292705877e-10;
  double p = 1.0 / 6227020800.0;
  p = p * r; p = p + 1.0 / 479001600.0;
  p = p * r; p = p + 1.0 / 39916800.0;
  p = p * r; p = p + 1.0 / 3628800.0;
  p = p * r; p = p + 1.0 / 362880.0;
  p = p * r; p = p + 1.0 / 40320.0;
  p = p * r; p = p + 1.0 / 5040.0;
  p = p * r; p = p + 1.0 / 720.0;
  p = p * r; p = p + 1.0 / 120.0;
  p = p * r; p = p + 1.0 / 24.0;
  p = p * r; p = p + 1.0 / 6.0;
  p = p * r; p = p + 1.0 / 2.0;
  p = p * r; p = p + 1.0;
  p = p * r; p = p + 1.0;
  return __builtin_ldexp(p, (int)k);
}

template <int EPL, int K, int J>
__device__ __forceinline__ void bitonic_step(uint32_t (&key)[EPL], int lane) {
  constexpr int NKP = 64 * EPL;
  // element v = lane * EPL + t; a step compares v with v ^ J inside blocks of size K (descending where (v & K) == 0)
  if constexpr (J >= EPL) {
    constexpr int DL = J / EPL;                                     // partner lane = lane ^ DL
    const bool lower = (lane & DL) == 0;
    const bool desc = (K >= NKP) ? true : ((lane & (K / EPL)) == 0);
    const bool want_max = lower == desc;
#pragma unroll
    for (int t = 0; t < EPL; t++) {
      uint32_t o, own = key[t];
      if constexpr (DL >= 16) pair_of_u32<DL>(own, own, o);        // (the maximum and the minimum do not ask which is whose)
      else o = lane_xor_u32<DL>(own);
      const uint32_t mx = own > o ? own : o, mn = own > o ? o : own;
      key[t] = want_max ? mx : mn;
    }
  } else {
#pragma unroll
    for (int t = 0; t < EPL; t++) {
      if ((t & J) == 0) {
        const uint32_t a = key[t], b = key[t | J];
        const uint32_t mx = a > b ? a : b, mn = a > b ? b : a;
        if constexpr (K < EPL) {
          const bool desc = (t & K) == 0;                           // compile-time
          key[t] = desc ? mx : mn;
          key[t | J] = desc ? mn : mx;
        } else {
          const bool desc = (K >= NKP) ? true : ((lane & (K / EPL)) == 0);
          key[t] = desc ? mx : mn;
          key[t | J] = desc ? mn : mx;
        }
      }
    }
  }
}
template <int EPL, int K, int J>
__device__ __forceinline__ void bitonic_inner(uint32_t (&key)[EPL], int lane) {
  bitonic_step<EPL, K, J>(key, lane);
  if constexpr (J > 1) bitonic_inner<EPL, K, J / 2>(key, lane);
}
template <int EPL, int K>
__device__ __forceinline__ void bitonic_sort_desc(uint32_t (&key)[EPL], int lane) {
  bitonic_inner<EPL, K, K / 2>(key, lane);
  if constexpr (K < 64 * EPL) bitonic_sort_desc<EPL, K * 2>(key, lane);
}

// =============================================================================================
// A whole row of at most 64 W columns in one wavefront: lane l holds columns l, l + 64, ...  Same arithmetic as
// block_select_wave_kernel with W columns per lane, and the result stays a map of W 64-bit words: bit j = column j is kept.
// =============================================================================================
// Pooled score of row `qrow` (D elements) against a pooled K row, by the four lanes of a group: lane `part` takes the
// 16-byte pieces part, part + 4, ...  Products of two 16-bit floats and their sums are exact in binary64, so the order of
// the additions is free.  Every lane of the group returns the rounded, scaled score.
template <int D, int DT>
__device__ __forceinline__ uint16_t pooled_score_4lanes(const uint16_t *__restrict__ qrow, const uint16_t *__restrict__ krow, int part) {
#pragma clang fp contract(off)
  uint4 qv[D / 32], kv[D / 32];
#pragma unroll
  for (int t = 0; t < D / 32; t++) {
    qv[t] = *(const uint4 *)(qrow + 8 * (part + 4 * t));
    kv[t] = *(const uint4 *)(krow + 8 * (part + 4 * t));
  }
  double acc = 0.0;
#pragma unroll
  for (int t = 0; t < D / 32; t++) {
    const uint32_t qw[4] = {qv[t].x, qv[t].y, qv[t].z, qv[t].w}, kw[4] = {kv[t].x, kv[t].y, kv[t].z, kv[t].w};
#pragma unroll
    for (int e = 0; e < 4; e++) {
      acc = __builtin_fma((double)elem_to_f32<DT>((uint16_t)(qw[e] & 0xffffu)), (double)elem_to_f32<DT>((uint16_t)(kw[e] & 0xffffu)), acc);
      acc = __builtin_fma((double)elem_to_f32<DT>((uint16_t)(qw[e] >> 16)), (double)elem_to_f32<DT>((uint16_t)(kw[e] >> 16)), acc);
    }
  }
  acc = group_sum_f64<4>(acc);
  const float sm_scale = (D == 64) ? 0.125f : 0.088388347648318447f;  // fp32(D^-0.5)
  const float s1 = elem_to_f32<DT>(f64_to_elem_fast<DT>(acc));
  return f64_to_elem_fast<DT>((double)s1 * (double)sm_scale);
}

// sc[t]: the score of column 64 t + lane, -inf where the column is masked (beyond nk, dissimilar K block, causal).
// k_dead[t]: that column is a dissimilar K block (kept in every row).
template <int DT, int W>
__device__ __forceinline__ void select_row(uint64_t (&map)[W], const float (&sc)[W], const bool (&k_dead)[W], bool by_topk, float level,
                                           int nk, int causal_lim, bool row_forced, bool sink, int lane) {
#pragma clang fp contract(off)
  constexpr int LOW = W == 1 ? 6 : 7;                   // log2(64 W)
  static_assert(W == 1 || W == 2, "columns per lane");
  float lmax = sc[0];
#pragma unroll
  for (int t = 1; t < W; t++) lmax = fmaxf(lmax, sc[t]);
  const float mx = wave_max_f32(lmax);
  double ev[W], part = 0.0;
#pragma unroll
  for (int t = 0; t < W; t++) {
    ev[t] = (sc[t] == -INFINITY) ? 0.0 : cexp((double)sc[t] - (double)mx);
    part = part + ev[t];
  }
  const double total = wave_tree_sum_f64(part);
  uint32_t okey[W];
#pragma unroll
  for (int t = 0; t < W; t++) {
    double p = ev[t] / total;
    if (!__builtin_isfinite(p)) p = 0.0;
    const int j = 64 * t + lane;
    okey[t] = j < nk ? (((uint32_t)f64_to_elem_fast<DT>(p) << 16) | (0xffffu - (uint32_t)j)) : 0u;
  }
  int n;
  uint32_t kth = 0u;
  if (by_topk) {
    const float t = level * (float)nk;                  // binary32 product, truncated (utils.py:405)
    n = (int)fminf(fmaxf(t, 0.f), 64.f * W);
    if (n <= 0) n = 1;                                  // utils.py:289
    if (n < nk) {
      // n-th largest key, bit by bit (bits 31 and 30 are clear, 15..LOW are set in every real key); a candidate that exactly
      // n keys reach selects the same set
      uint32_t T = 0u;
      bool exact = false;
      auto try_bit = [&](int bit) {
        const uint32_t cand = T | (1u << bit);
        int cnt = 0;
#pragma unroll
        for (int t = 0; t < W; t++) cnt += __builtin_popcountll(__ballot(okey[t] >= cand));
        if (cnt >= n) T = cand;
        exact = cnt == n;
      };
#pragma unroll 1
      for (int bit = 29; bit >= 16 && !exact; bit--) try_bit(bit);
      if (!exact) {
        T |= 0xffffu & ~((1u << LOW) - 1u);
#pragma unroll 1
        for (int bit = LOW - 1; bit >= 0 && !exact; bit--) try_bit(bit);
      }
      kth = T;
    }
  } else {
    uint32_t key[W];
#pragma unroll
    for (int t = 0; t < W; t++) key[t] = okey[t];
    bitonic_sort_desc<W, 2>(key, lane);                 // sorted position of key[t] is lane * W + t
    // cdf[v] = T(sum_{u<=v} p_sorted[u]);  n = #{v < nk : cdf[v] <= threshold}  (utils.py:398-403).  fp16 probabilities are multiples of
    // 2^-24, so their sums are exact in any order.  bf16 ones reach further down than binary64 holds beside 1: probabilities below about
    // 2^-45 of the sum can be rounded, here and in the selection kernel in another order (with two columns per lane `run - own`, too).
    // That shows only if it carries the sum across a rounding tie of T that sits at the threshold.
    double own = 0.0;
#pragma unroll
    for (int t = 0; t < W; t++) own += (double)elem_to_f32<DT>((uint16_t)(key[t] >> 16));
    double run = own;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const uint64_t u = __builtin_bit_cast(uint64_t, run);
      const uint32_t lo = (uint32_t)__shfl_up((int)(uint32_t)u, o, SPG_WAVE), hi = (uint32_t)__shfl_up((int)(uint32_t)(u >> 32), o, SPG_WAVE);
      const double before = __builtin_bit_cast(double, ((uint64_t)hi << 32) | lo);
      run = lane >= o ? run + before : run;
    }
    n = 0;
    if constexpr (W > 1) run -= own;                    // of the lanes before this one
#pragma unroll
    for (int t = 0; t < W; t++) {
      if constexpr (W > 1) run += (double)elem_to_f32<DT>((uint16_t)(key[t] >> 16));
      const float cdfv = elem_to_f32<DT>(f64_to_elem<DT>(run));
      n += __builtin_popcountll(__ballot(lane * W + t < nk && (double)cdfv <= (double)level));
    }
    if (n <= 0) n = 1;                                  // utils.py:289
    if (n < nk) {                                       // wavefront-uniform
      uint32_t mine = key[0];
#pragma unroll
      for (int t = 1; t < W; t++) mine = (n - 1) % W == t ? key[t] : mine;
      kth = (uint32_t)__shfl((int)mine, (n - 1) / W, SPG_WAVE);
    }
  }
#pragma unroll
  for (int t = 0; t < W; t++) {
    const int j = 64 * t + lane;
    bool f = false;
    if (j < nk) {
      f = row_forced || okey[t] >= kth || k_dead[t];
      if (j >= causal_lim) f = false;
      if (sink && j == 0) f = true;
    }
    map[t] = __ballot(f);
  }
}

}  // namespace spg
