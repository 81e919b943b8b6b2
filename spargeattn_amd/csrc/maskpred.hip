// Sparse-mask prediction and INT8 Q/K quantisation for gfx950.
//
// Kernels (one 16-byte load per lane, 64-lane wavefront reductions; the K mean and the pooling / quantisation kernels run
// at the rates the machine gives a bare read and a bare 2-bytes-in / 1-byte-out copy, the selection is bound by the
// exact arithmetic it carries):
//   km_partial / km_final      K column mean                          (spas_sage_attn/core.py:119-120)
//   pool_sim_quant             pool + self-similarity + INT8 quant    (spas_sage_attn/utils.py:161-214, 89-159)
//   block_select_wave / block_select   compressed QK^T softmax, top-k / CDF selection, block map, delta LUT: pooled
//                              scores on the binary64 matrix unit and one wavefront per row with the row in registers
//                              (nk <= 2048), one workgroup per row beyond
//                                                                     (spas_sage_attn/utils.py:386-420, 54-87, 282-316)
//   map_to_lut                 user block mask -> LUT                 (spas_sage_attn/utils.py:54-87)
//
// Arithmetic contract: reductions whose addends are exactly representable run in binary64 (exact, hence
// order independent); every tensor the reference materialises in the input dtype is rounded exactly once
// (round-to-nearest-even, straight from binary64); fp32 quantisation steps use IEEE divide / sqrt; the
// compressed softmax uses a fixed binary64 operation sequence and a fixed summation tree.  This file must be
// compiled with -ffp-contract=off.
#include "select_row.h"
#include "stage_bodies.h"

#include <atomic>

namespace spg {

// =============================================================================================
// K column mean
// =============================================================================================
template <int D, int DT>
__global__ __launch_bounds__(256) void km_partial_kernel(const uint16_t *__restrict__ k, const Strides ks, int H,
                                                         double *__restrict__ part, int N, int rows_per_chunk) {
  __shared__ __align__(16) unsigned char smem[km_partial_lds<D>()];
  km_partial_body<D, DT>(k, ks, H, part, N, rows_per_chunk, blockIdx.x, gridDim.x, blockIdx.y, smem);
}

// One workgroup per (batch, head), blockDim = (D, 8): eight threads share a column's partial sums (exact, so the order of
// the additions is free), thread (d, 0) adds the eight sub-sums and rounds.
template <int DT>
__global__ void km_final_kernel(const double *__restrict__ part, uint16_t *__restrict__ km, int nchunk, int D, int N) {
  __shared__ double s_sub[8][128];
  const int bh = blockIdx.x, d = threadIdx.x, y = threadIdx.y;
  double s = 0.0;
#pragma unroll 4
  for (int i = y; i < nchunk; i += 8) s += part[((size_t)bh * nchunk + i) * D + d];
  s_sub[y][d] = s;
  __syncthreads();
  if (y == 0) {
    double t = 0.0;
#pragma unroll
    for (int u = 0; u < 8; u++) t += s_sub[u][d];
    km[(size_t)bh * D + d] = f64_to_elem<DT>(t / (double)N);
  }
}

// Self-test of div_by: divisor number i is a hash of (seed, i) with exponent in [-40, 40); every finite 16-bit
// numerator of both element types with |a| >= 2^-100 and 2^-100 <= |a/b| <= 2^100 is divided both ways.  counts[0] += comparisons,
// counts[1] += differing bit patterns other than a differently signed zero.
__global__ __launch_bounds__(256) void div_selftest_kernel(unsigned long long *counts, int n_div, uint32_t seed) {
  auto hash32 = [](uint32_t x) { x ^= x >> 16; x *= 0x7feb352du; x ^= x >> 15; x *= 0x846ca68bu; x ^= x >> 16; return x; };
  const uint32_t bi = blockIdx.x * 256u + threadIdx.x;
  if (bi >= (uint32_t)n_div) return;
  const uint32_t h = hash32(bi * 2654435761u + seed);
  const int ex = (int)(hash32(h) % 80u) - 40;
  const float b = __builtin_bit_cast(float, ((uint32_t)(127 + ex) << 23) | (h & 0x7fffffu));
  const float r = exact_rcp(b);
  unsigned long long bad = 0, tot = 0;
  for (uint32_t pat = 0; pat < 65536u; pat++) {
#pragma unroll
    for (int kind = 0; kind < 2; kind++) {
      const float a = kind == 0 ? elem_to_f32<1>((uint16_t)pat) : elem_to_f32<0>((uint16_t)pat);
      if (!__builtin_isfinite(a) || (__builtin_fabsf(a) < 0x1p-100f && a != 0.0f)) continue;
      const float want = a / b, got = div_by(a, b, r);
      const float mag = __builtin_fabsf(want);
      if (want != 0.0f && !(mag >= 0x1p-100f && mag <= 0x1p100f)) continue;   // outside the range the callers use
      tot++;
      if (__builtin_bit_cast(uint32_t, want) != __builtin_bit_cast(uint32_t, got) && !(want == 0.0f && got == 0.0f)) bad++;
    }
  }
  atomicAdd(&counts[0], tot);
  atomicAdd(&counts[1], bad);
}

// pool + sim + INT8 quantisation: one workgroup per (128 rows, b*h)
template <int BS, int D, int DT, bool HAS_MEAN, bool WITH_POOL, int QR = BS>
__global__ __launch_bounds__(256) void pool_sim_quant_kernel(const uint16_t *__restrict__ x, const Strides xs,
                                                             const uint16_t *__restrict__ km,
                                                             uint16_t *__restrict__ pool, uint8_t *__restrict__ sim,
                                                             int8_t *__restrict__ xq, float *__restrict__ scale,
                                                             const float *__restrict__ simthr, int H, int N, int nb) {
  __shared__ __align__(16) unsigned char smem[WITH_POOL ? psq_lds<BS, D>() : 16];
  float thr = 0.f;
  if constexpr (WITH_POOL) thr = simthr[blockIdx.y % H];
  psq_body<BS, D, DT, HAS_MEAN ? MEAN_GIVEN : MEAN_NONE, WITH_POOL, QR>(x, xs, km, nullptr, 0, pool, sim, xq, scale, thr, H, N, nb,
                                                                        blockIdx.x, blockIdx.y, smem);
}

// =============================================================================================
// block_select: one workgroup per (R consecutive q block rows, b*h).
// Phase 1 computes the R x nk pooled scores with every pooled-K row read ONCE for the R rows (one lane per
// column, binary64 accumulation in the fixed order d = 0..D-1); phase 2 handles the rows one after the other:
// softmax, stable descending sort, top-k / CDF count, block-map row, delta LUT.
// dynamic LDS: R*D*8 (pooled Q as doubles) + R*nkp*4 (scores) + 12*nkp (per-row work area).
// =============================================================================================
template <int D, int DT, int R>
__global__ __launch_bounds__(256) void block_select_kernel(
    const uint16_t *__restrict__ pool_q, const uint8_t *__restrict__ sim_q, const uint16_t *__restrict__ pool_k,
    const uint8_t *__restrict__ sim_k, const bool by_topk, const Hyper level, int is_causal,
    int sink, int32_t *__restrict__ lut, int32_t *__restrict__ valid, int32_t *__restrict__ valid_out, uint8_t *__restrict__ bmap, int H, int Hkv, int nq,
    int nk, int nkp) {
  extern __shared__ __align__(16) unsigned char smem[];
  double *s_pq = (double *)smem;                                   // [R][D]
  float *s_scores = (float *)(smem + (size_t)R * D * 8);           // [R][nkp]
  unsigned char *work = smem + (size_t)R * D * 8 + (size_t)R * nkp * 4;
  double *e_buf = (double *)work;                      // [nkp] exp values        (step 1)
  uint32_t *skey = (uint32_t *)work;                   // [nkp] sorted keys       (step 2, aliases e_buf)
  int32_t *s_idx = (int32_t *)(work + 4 * (size_t)nkp);    // [nkp] compact indices (step 3, aliases e_buf)
  uint32_t *okey = (uint32_t *)(work + 8 * (size_t)nkp);   // [nkp] keys in column order
  __shared__ float s_wmax[4];
  __shared__ double s_wsum[4];
  __shared__ double s_tsum[256];
  __shared__ int s_tmp[256];
  __shared__ int s_n;

  const int i0 = blockIdx.x * R, bh = blockIdx.y, h = bh % H, tid = threadIdx.x;
  const int rows = min(R, nq - i0);
  for (int t = tid; t < R * D; t += 256) {
    const int row = t / D;
    s_pq[t] = row < rows ? (double)elem_to_f32<DT>(pool_q[((size_t)bh * nq + i0 + row) * D + (t % D)]) : 0.0;
  }
  __syncthreads();

  const float sm_scale = (D == 64) ? 0.125f : 0.088388347648318447f;  // fp32(D^-0.5)
  // grouped K/V heads: query head h is scored against the pooled blocks of K head h / (H / Hkv)
  const int bhk = (bh / H) * Hkv + h / (H / Hkv);
  const uint16_t *pk_base = pool_k + (size_t)bhk * nk * D;
  const uint8_t *simk = sim_k + (size_t)bhk * nk;

  // ---- phase 1: scores.  Products of two 16-bit floats are exact in binary64, so fma == multiply-then-add. ----
  for (int j = tid; j < nk; j += 256) {
    double acc[R];
#pragma unroll
    for (int row = 0; row < R; row++) acc[row] = 0.0;
    const uint4 *krow = (const uint4 *)(pk_base + (size_t)j * D);
#pragma unroll 2
    for (int cch = 0; cch < D / 8; cch++) {
      const uint4 v = krow[cch];
      const uint32_t w[4] = {v.x, v.y, v.z, v.w};
      double kd[8];
#pragma unroll
      for (int e = 0; e < 8; e++)
        kd[e] = (double)elem_to_f32<DT>((uint16_t)((e & 1) ? (w[e >> 1] >> 16) : (w[e >> 1] & 0xffffu)));
#pragma unroll
      for (int row = 0; row < R; row++) {
        const double *q = s_pq + row * D + cch * 8;
#pragma unroll
        for (int e = 0; e < 8; e++) acc[row] = __builtin_fma(q[e], kd[e], acc[row]);
      }
    }
    const bool dead_col = simk[j] == 0;
#pragma unroll
    for (int row = 0; row < R; row++) {
      const float s1 = elem_to_f32<DT>(f64_to_elem<DT>(acc[row]));
      float s2 = elem_to_f32<DT>(f64_to_elem<DT>((double)s1 * (double)sm_scale));
      if (dead_col || (is_causal && j >= 2 * (i0 + row + 1))) s2 = -INFINITY;
      s_scores[(size_t)row * nkp + j] = s2;
    }
  }
  __syncthreads();

  // ---- phase 2: one row at a time ------------------------------------------------------------------------
  for (int row = 0; row < rows; row++) {
    const int i = i0 + row;
    const int causal_lim = is_causal ? min(nk, 2 * (i + 1)) : nk;
    const float *s_score = s_scores + (size_t)row * nkp;

    float lmax = -INFINITY;
    for (int j = tid; j < nk; j += 256) lmax = fmaxf(lmax, s_score[j]);
    lmax = wave_max_f32(lmax);
    if ((tid & 63) == 0) s_wmax[tid >> 6] = lmax;
    __syncthreads();
    const float mx = fmaxf(fmaxf(s_wmax[0], s_wmax[1]), fmaxf(s_wmax[2], s_wmax[3]));

    // exp, then the fixed summation tree: lane l of ONE wavefront adds e[l], e[l+64], ... in order, followed by an
    // xor butterfly (32 .. 1)
    for (int j = tid; j < nk; j += 256) {
      const float s2 = s_score[j];
      e_buf[j] = (s2 == -INFINITY) ? 0.0 : cexp((double)s2 - (double)mx);
    }
    __syncthreads();
    if (tid < 64) {
      double part = 0.0;
      for (int j = tid; j < nk; j += 64) part = part + e_buf[j];
      part = wave_tree_sum_f64(part);
      if (tid == 0) s_wsum[0] = part;
    }
    __syncthreads();
    const double total = s_wsum[0];

    // probabilities -> sortable keys (value bits, then lower index first)
    for (int j = tid; j < nk; j += 256) {
      double p = e_buf[j] / total;
      if (!__builtin_isfinite(p)) p = 0.0;
      const uint32_t bits = f64_to_elem<DT>(p);
      okey[j] = (bits << 16) | (0xffffu - (uint32_t)j);
    }
    __syncthreads();
    for (int j = tid; j < nkp; j += 256) skey[j] = (j < nk) ? okey[j] : 0u;
    __syncthreads();

    // bitonic sort, descending
    for (int k = 2; k <= nkp; k <<= 1) {
      for (int lj = __builtin_ctz(k) - 1; lj >= 0; lj--) {     // compare distance j = 2^lj
        const int j = 1 << lj;
        for (int t = tid; t < nkp / 2; t += 256) {
          const int lo = ((t >> lj) << (lj + 1)) | (t & (j - 1));
          const int hi = lo | j;
          const bool desc = (lo & k) == 0;
          const uint32_t a = skey[lo], b = skey[hi];
          if ((a < b) == desc) { skey[lo] = b; skey[hi] = a; }
        }
        __syncthreads();
      }
    }

    // how many to keep
    long long n;
    if (by_topk) {
      const float t = level.at(h) * (float)nk;     // binary32 product, truncated (utils.py:405)
      n = (long long)t;
    } else {
      // cdf[i] = T(sum_{u<=i} p_sorted[u]);  n = #{i < nk : cdf[i] <= threshold}  (utils.py:398-403)
      const int seg = nkp / 256;
      const int p0 = tid * seg;
      double lsum = 0.0;
      for (int u = 0; u < seg; u++) lsum += (double)elem_to_f32<DT>((uint16_t)(skey[p0 + u] >> 16));
      s_tsum[tid] = lsum;
      __syncthreads();
      double run = 0.0;
      for (int u = 0; u < tid; u++) run += s_tsum[u];
      const double thr = (double)level.at(h);
      int cnt = 0;
      for (int u = 0; u < seg; u++) {
        run += (double)elem_to_f32<DT>((uint16_t)(skey[p0 + u] >> 16));
        const float cdfv = elem_to_f32<DT>(f64_to_elem<DT>(run));
        if (p0 + u < nk && (double)cdfv <= thr) cnt++;
      }
      cnt = wave_sum_i32(cnt);
      if (tid == 0) s_n = 0;
      __syncthreads();
      if ((tid & 63) == 0) atomicAdd(&s_n, cnt);
      __syncthreads();
      n = s_n;
    }
    if (n <= 0) n = 1;                              // utils.py:289
    const uint32_t kth = (n >= nk) ? 0u : skey[n - 1];
    __syncthreads();                                // skey is dead from here

    // block map row and LUT
    const bool row_forced = sim_q[(size_t)bh * nq + i] == 0;
    auto flag = [&](int j) -> bool {
      bool f = row_forced || (okey[j] >= kth) || (simk[j] == 0);
      if (j >= causal_lim) f = false;
      if (sink && j == 0) f = true;
      return f;
    };
    const size_t row_off = ((size_t)bh * nq + i) * nk;
    if (bmap != nullptr)
      for (int j = tid; j < nk; j += 256) bmap[row_off + j] = flag(j) ? 1 : 0;
    emit_lut<256>(flag, nk, nkp, s_idx, s_tmp, lut + row_off, valid + (size_t)bh * nq + i);
    __syncthreads();                                // the work area is reused by the next row
    if (valid_out != nullptr && tid == 0) valid_out[(size_t)bh * nq + i] = valid[(size_t)bh * nq + i];
  }
}

// A probability e / total as a 16-bit pattern, from e * (1 / total), which is within two units in the last place of the quotient:
// through binary32, the two agree unless the product lands exactly on a rounding tie of the 16-bit format or outside its normal
// range, and those elements take the division and the exact conversion.
template <int DT> __device__ __forceinline__ uint32_t probability_bits(double e, double total, double rtotal) {
  const float pr = (float)(e * rtotal);
  const uint32_t pb = __builtin_bit_cast(uint32_t, pr);    // probabilities are non-negative
  constexpr uint32_t DROP = DT == 1 ? 16u : 13u, LOWM = (1u << DROP) - 1u, TIE = 1u << (DROP - 1u);
  constexpr uint32_t LO = DT == 1 ? 0x00800000u : 0x38800000u;     // smallest normal of the format
  const bool safe = pb == 0u || (pb >= LO && pb <= 0x3f800000u && (pb & LOWM) != TIE);
  if (safe) return f32_to_elem<DT>(pr);
  double p = e / total;
  if (!__builtin_isfinite(p)) p = 0.0;
  return f64_to_elem<DT>(p);
}

// Top-k needs the n-th largest key only, not the order: build it bit by bit, the largest T with #{key >= T} >= n.  Keys are
// distinct, probabilities are <= 1 (bits 31 and 30 of a key are clear) and bits 15 .. log2(64 EPL) are set in every real key (they
// hold 0xFFFF - column).  A candidate that exactly n keys reach selects the same set as the n-th largest key itself, so the
// search stops there.
template <int EPL> __device__ __forceinline__ uint32_t nth_largest_key(const uint32_t (&okey)[EPL], int n) {
  constexpr int LOW = 31 - __builtin_clz((unsigned)(64 * EPL));
  uint32_t T = 0u;
  bool exact = false;                                      // wavefront-uniform
  auto try_bit = [&](int bit) {
    const uint32_t cand = T | (1u << bit);
    int cnt = 0;
#pragma unroll
    for (int tt = 0; tt < EPL; tt++) cnt += __builtin_popcountll(__ballot(okey[tt] >= cand));
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
  return T;
}

// =============================================================================================
// block_select, wavefront-per-row variant (nk <= 2048).
// Phase 1 computes the scores of 16 pooled-Q rows against all pooled-K rows on the matrix unit in binary64
// (v_mfma_f64_16x16x4_f64: operands are delivered once per 1024 multiply-adds instead of once per multiply-add) and
// leaves them in LDS as 16-bit patterns.  Phase 2 gives each of the eight wavefronts its own rows (one of R = 8, two of
// R = 16) and keeps a whole row
// in registers (EPL = nkp / 64 columns per lane): no workgroup barrier, the stable descending sort is a bitonic network
// whose short-distance steps are register-local and whose long-distance steps are lane exchanges.
// dynamic LDS: R*nkp*2 (scores) + 8*nkp*2 (per-wave index list) + 8*64*8 (lane sums).
// =============================================================================================
template <int D, int DT, int NW, int EPL, bool DUAL, int R>
__global__ __launch_bounds__(64 * NW, (!DUAL && NW == 8) ? 2 : 1) void block_select_wave_kernel(
    const uint16_t *__restrict__ pool_q, const uint8_t *__restrict__ sim_q, const uint16_t *__restrict__ pool_k,
    const uint8_t *__restrict__ sim_k, const bool by_topk, const Hyper level, int is_causal,
    int sink, int32_t *__restrict__ lut, int32_t *__restrict__ valid, int32_t *__restrict__ valid_out, uint8_t *__restrict__ bmap, int H, int Hkv, int nq,
    int nk) {
  // R rows per workgroup; phase 1 computes 16 x 16 score tiles on the matrix unit, of which R = 8 uses the first 8 rows
  static_assert(R == 16 || R == 8, "rows per workgroup");
  constexpr int NKP = 64 * EPL;
  static_assert(NW == 8 || NW == 16, "wavefronts per workgroup");
  extern __shared__ __align__(16) unsigned char smem[];
  uint16_t *s_scores = (uint16_t *)smem;                                      // [R][NKP] scores as 16-bit patterns
  uint16_t *s_idx_all = (uint16_t *)(smem + (size_t)R * NKP * 2);             // [NW][NKP] (column indices are below 2048)
  double *s_lsum_all = (double *)(smem + (size_t)R * NKP * 2 + NW * (size_t)NKP * 2);   // [NW][64]

  // Causal rows get heavier with the row index.  Workgroups that differ by 8 in blockIdx.y tend to share a CU (ids are
  // dealt round-robin over 8 XCDs, then over the CUs of an XCD), so the row-group index is rotated by a quarter of
  // the grid per such step: a CU then holds a mix of light and heavy row groups.
  const int bx = (int)((blockIdx.x + (blockIdx.y >> 3) * (gridDim.x >> 2)) % gridDim.x);
  const int i0 = bx * R, bh = blockIdx.y, h = bh % H, tid = threadIdx.x;
  const int rows = min(R, nq - i0);
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);

  const float sm_scale = (D == 64) ? 0.125f : 0.088388347648318447f;  // fp32(D^-0.5)
  // grouped K/V heads: query head h is scored against the pooled blocks of K head h / (H / Hkv)
  const int bhk = (bh / H) * Hkv + h / (H / Hkv);
  const uint16_t *pk_base = pool_k + (size_t)bhk * nk * D;
  const uint8_t *simk = sim_k + (size_t)bhk * nk;

  // ---- phase 1: the 16 x nk pooled scores in binary64 on the matrix unit (v_mfma_f64_16x16x4_f64) --------------------
  // Products of two 16-bit floats are exact in binary64 and so are their partial sums (the contract's domain), so the
  // sum does not depend on the order of the terms: a tile of 16 rows x 16 columns accumulates the D dimensions four at a
  // time.  Lane l = 16 g + c supplies A[c][g] (pooled Q row c) and B[g][c] (pooled K column c) of each step and receives
  // rows g, g + 4, g + 8, g + 12 of column c.  Step s pairs lane group g with dimension 32 (s / 8) + 8 g + (s % 8): every lane
  // then consumes the eight values of one 16-byte load in eight consecutive steps.
  {
    typedef double d4_t __attribute__((ext_vector_type(4)));
    constexpr int NL = D / 32;                    // 16-byte loads per row and lane
    const int c = lane & 15, g = lane >> 4;
    double qa[D / 4];
    {
      const bool row_ok = c < rows;
      const uint16_t *qrow = pool_q + ((size_t)bh * nq + i0 + (row_ok ? c : 0)) * D + 8 * g;
#pragma unroll
      for (int t = 0; t < NL; t++) {
        const uint4 v = row_ok ? *(const uint4 *)(qrow + 32 * t) : make_uint4(0, 0, 0, 0);
        const uint32_t w[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
        for (int e = 0; e < 8; e++)
          qa[8 * t + e] = (double)elem_to_f32<DT>((uint16_t)((e & 1) ? (w[e >> 1] >> 16) : (w[e >> 1] & 0xffffu)));
      }
    }
    // columns at or beyond j_live are masked for every row of this workgroup: they get -inf without any arithmetic
    const int j_live = is_causal ? min(nk, 2 * (i0 + rows)) : nk;
    constexpr uint16_t NEG_INF = DT == 1 ? 0xff80u : 0xfc00u;
    const int n_tiles = NKP / 16, live_tiles = (j_live + 15) / 16;
    auto load_k = [&](int ct, uint4 (&raw)[NL]) __attribute__((always_inline)) {
      const int j = min(16 * ct + c, nk - 1);    // columns beyond nk re-read the last one and are masked below
      const uint16_t *krow = pk_base + (size_t)j * D + 8 * g;
#pragma unroll
      for (int t = 0; t < NL; t++) raw[t] = *(const uint4 *)(krow + 32 * t);
    };
    auto finish = [&](int ct, const d4_t &acc) __attribute__((always_inline)) {
      const int j = 16 * ct + c;
      const bool dead = j >= nk || simk[min(j, nk - 1)] == 0;
#pragma unroll
      for (int v = 0; v < R / 4; v++) {
        const int row = g + 4 * v;
        const float a1 = elem_to_f32<DT>(f64_to_elem_fast<DT>(acc[v]));
        uint16_t a2 = f64_to_elem_fast<DT>((double)a1 * (double)sm_scale);
        if (dead || (is_causal && j >= 2 * (i0 + row + 1))) a2 = NEG_INF;
        s_scores[(size_t)row * NKP + j] = a2;
      }
    };
    // DUAL: two column tiles per trip (two independent accumulator chains), for the long rows that leave a SIMD only two
    // wavefronts; otherwise one (128 registers per lane, four wavefronts per SIMD keep the matrix unit busy instead).
    // The next trip's pooled-K rows are in flight meanwhile.
    constexpr int STEP = DUAL ? 2 * NW : NW;
    uint4 ra[NL], rb[DUAL ? NL : 1];
    int ct = wave;
    if (ct < live_tiles) {
      load_k(ct, ra);
      if constexpr (DUAL) load_k(min(ct + NW, live_tiles - 1), rb);
    }
#pragma unroll 1
    for (; ct < live_tiles; ct += STEP) {
      uint4 ka[NL], kb[DUAL ? NL : 1];
#pragma unroll
      for (int t = 0; t < NL; t++) { ka[t] = ra[t]; if constexpr (DUAL) kb[t] = rb[t]; }
      const bool two = DUAL && ct + NW < live_tiles;         // wavefront-uniform
      if (ct + STEP < live_tiles) {
        load_k(ct + STEP, ra);
        if constexpr (DUAL) load_k(min(ct + STEP + NW, live_tiles - 1), rb);
      }
      d4_t acc_a = {0.0, 0.0, 0.0, 0.0}, acc_b = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
      for (int t = 0; t < NL; t++) {
        const uint32_t wa[4] = {ka[t].x, ka[t].y, ka[t].z, ka[t].w};
#pragma unroll
        for (int e = 0; e < 8; e++) {
          const double xa = (double)elem_to_f32<DT>((uint16_t)((e & 1) ? (wa[e >> 1] >> 16) : (wa[e >> 1] & 0xffffu)));
          acc_a = __builtin_amdgcn_mfma_f64_16x16x4f64(qa[8 * t + e], xa, acc_a, 0, 0, 0);
          if constexpr (DUAL) {
            const uint32_t wb[4] = {kb[t].x, kb[t].y, kb[t].z, kb[t].w};
            const double xb = (double)elem_to_f32<DT>((uint16_t)((e & 1) ? (wb[e >> 1] >> 16) : (wb[e >> 1] & 0xffffu)));
            acc_b = __builtin_amdgcn_mfma_f64_16x16x4f64(qa[8 * t + e], xb, acc_b, 0, 0, 0);
          }
        }
      }
      finish(ct, acc_a);
      if (two) finish(ct + NW, acc_b);
    }
    // dead column tiles
    for (int t2 = live_tiles + wave; t2 < n_tiles; t2 += NW) {
      const int j = 16 * t2 + c;
#pragma unroll
      for (int v = 0; v < R / 4; v++) s_scores[(size_t)(g + 4 * v) * NKP + j] = NEG_INF;
    }
  }
  __syncthreads();

  // ---- phase 2: wavefront `wave` owns rows wave, wave + NW, ...; lane l holds columns l, l + 64, ... ---------------
  uint16_t *s_idx = s_idx_all + wave * NKP;
  double *s_lsum = s_lsum_all + wave * 64;
  for (int row = wave; row < rows; row += NW) {
    const int i = i0 + row;
    const int causal_lim = is_causal ? min(nk, 2 * (i + 1)) : nk;
    const uint16_t *s_score = s_scores + (size_t)row * NKP;

    float sc[EPL];
    float lmax = -INFINITY;
#pragma unroll
    for (int t = 0; t < EPL; t++) {
      sc[t] = elem_to_f32<DT>(s_score[t * 64 + lane]);   // columns >= nk were written as -inf by phase 1
      lmax = fmaxf(lmax, sc[t]);
    }
    const float mx = wave_max_f32(lmax);

    // exp and the fixed summation tree: lane l adds e[l], e[l+64], ... in order, then an xor butterfly (32 .. 1)
    double ev[EPL];
    double part = 0.0;
#pragma unroll
    for (int t = 0; t < EPL; t++) {
      ev[t] = (sc[t] == -INFINITY) ? 0.0 : cexp((double)sc[t] - (double)mx);
      part = part + ev[t];
    }
    part = wave_tree_sum_f64(part);
    const double total = part;

    // probabilities -> sortable keys (value bits, then lower column first)
    const double rtotal = total > 0.0 ? 1.0 / total : 0.0;     // a row without a live column has e = 0 everywhere
    uint32_t okey[EPL], key[EPL];
#pragma unroll
    for (int t = 0; t < EPL; t++) {
      const int j = t * 64 + lane;
      okey[t] = j < nk ? ((probability_bits<DT>(ev[t], total, rtotal) << 16) | (0xffffu - (uint32_t)j)) : 0u;
      key[t] = okey[t];
    }
    // how many to keep, and the key of the last one kept
    long long n;
    uint32_t kth = 0u;
    if (by_topk) {
      const float t = level.at(h) * (float)nk;            // binary32 product, truncated (utils.py:405)
      n = (long long)t;
      if (n <= 0) n = 1;                              // utils.py:289
      if (n < nk) kth = nth_largest_key<EPL>(okey, (int)n);
    } else {
      bitonic_sort_desc<EPL, 2>(key, lane);           // sorted position of key[t] is lane * EPL + t
      // cdf[v] = T(sum_{u<=v} p_sorted[u]);  n = #{v < nk : cdf[v] <= threshold}  (utils.py:398-403)
      double lsum = 0.0;
#pragma unroll
      for (int t = 0; t < EPL; t++) lsum += (double)elem_to_f32<DT>((uint16_t)(key[t] >> 16));
      s_lsum[lane] = lsum;
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      __builtin_amdgcn_wave_barrier();
      double run = 0.0;
      for (int u = 0; u < lane; u++) run += s_lsum[u];
      const double thr = (double)level.at(h);
      int cnt = 0;
#pragma unroll
      for (int t = 0; t < EPL; t++) {
        run += (double)elem_to_f32<DT>((uint16_t)(key[t] >> 16));
        const float cdfv = elem_to_f32<DT>(f64_to_elem_fast<DT>(run));
        if (lane * EPL + t < nk && (double)cdfv <= thr) cnt++;
      }
      n = wave_sum_i32(cnt);
      __builtin_amdgcn_wave_barrier();
      if (n <= 0) n = 1;                              // utils.py:289
      if (n < nk) {                                   // wavefront-uniform
        const int pos = (int)n - 1, src = pos / EPL, tt = pos % EPL;
        uint32_t mine = key[0];
#pragma unroll
        for (int t = 1; t < EPL; t++) mine = (tt == t) ? key[t] : mine;
        kth = (uint32_t)__shfl((int)mine, src, SPG_WAVE);
      }
    }

    // block map row, ascending index list, delta LUT
    const bool row_forced = sim_q[(size_t)bh * nq + i] == 0;
    const size_t row_off = ((size_t)bh * nq + i) * nk;
    int base = 0;
#pragma unroll
    for (int t = 0; t < EPL; t++) {
      const int j = t * 64 + lane;
      bool f = false;
      if (j < nk) {
        f = row_forced || (okey[t] >= kth) || (simk[j] == 0);
        if (j >= causal_lim) f = false;
        if (sink && j == 0) f = true;
        if (bmap != nullptr) bmap[row_off + j] = f ? 1 : 0;
      }
      const unsigned long long m = __ballot(f);
      const int below = __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0));
      if (f) s_idx[base + below] = (uint16_t)j;
      base += __builtin_popcountll(m);
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
#pragma unroll
    for (int t = 0; t < EPL; t++) {
      const int pidx = t * 64 + lane;
      if (pidx < nk) {
        int v = 0;
        if (pidx < base) v = (int)s_idx[pidx] - (pidx ? (int)s_idx[pidx - 1] : 0);
        lut[row_off + pidx] = v;
      }
    }
    if (lane == 0) {
      valid[(size_t)bh * nq + i] = base;
      if (valid_out != nullptr) valid_out[(size_t)bh * nq + i] = base;
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();                  // the index list is reused by this wavefront's next row
  }
}

// =============================================================================================
// block_select, workgroup-per-row variant (nk <= 2048), for grids that leave most of the chip idle.
// A row alone is a chain of steps that wait for each other, so what counts is the length of that chain: of 14.9 us in the
// kernel above (one head, nk 278, CDF) the scores took 5.3 (three tiles behind one another on the matrix unit, half of each
// tile for rows that are not there), the sort of 512 keys in one wavefront 2.6, the running sums and their conversion 2.2.
// Launch of 139 such rows: 16.2 us there, 8.8 here; 64 rows of nk 1875, D=128, top-k: the call 210 -> 167.
// Here the eight (nk <= 256: four) wavefronts of a workgroup share every step that can be shared: four lanes to a score, P = EPL / NW
// columns per lane for exponentials and keys, a sort of 64 P keys per wavefront and the merge by rank (a binary search in each of
// the other sorted runs).  Only the running sums are one wavefront's, since their order is part of the result.
// =============================================================================================
template <int D, int DT, int EPL>
__global__ __launch_bounds__(EPL == 4 ? 256 : 512) void block_select_row_kernel(
    const uint16_t *__restrict__ pool_q, const uint8_t *__restrict__ sim_q, const uint16_t *__restrict__ pool_k,
    const uint8_t *__restrict__ sim_k, const bool by_topk, const Hyper level, int is_causal,
    int sink, int32_t *__restrict__ lut, int32_t *__restrict__ valid, int32_t *__restrict__ valid_out, uint8_t *__restrict__ bmap, int H, int Hkv, int nq,
    int nk) {
  constexpr int NKP = 64 * EPL, NW = EPL == 4 ? 4 : 8, NT = 64 * NW, P = EPL / NW, RUN = 64 * P;
  __shared__ uint16_t s_score[NKP];                     // scores as 16-bit patterns
  __shared__ double s_ev[NKP];                          // exponentials
  __shared__ __align__(16) uint32_t s_run[NKP];         // keys (top-k) or NW sorted runs of RUN keys (CDF)
  __shared__ __align__(16) uint32_t s_sorted[NKP];
  __shared__ double s_lsum[128];                        // 64 zeros, then the lane sums
  __shared__ uint64_t s_map[EPL];
  __shared__ uint32_t s_kth;

  const int i = blockIdx.x, bh = blockIdx.y, h = bh % H, tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const float sm_scale = (D == 64) ? 0.125f : 0.088388347648318447f;  // fp32(D^-0.5)
  const int bhk = (bh / H) * Hkv + h / (H / Hkv);
  const uint16_t *pk_base = pool_k + (size_t)bhk * nk * D;
  const uint8_t *simk = sim_k + (size_t)bhk * nk;
  const int causal_lim = is_causal ? min(nk, 2 * (i + 1)) : nk;
  constexpr uint16_t NEG_INF = DT == 1 ? 0xff80u : 0xfc00u;

  // ---- scores: lane `part` of a group of four takes the 16-byte pieces part, part + 4, ...; products of two 16-bit floats and
  // their sums are exact in binary64, so the order of the additions is free
  {
    constexpr int NL = D / 32, COLS = NT / 4;           // columns per trip
    const int part = tid & 3, c = tid >> 2;
    auto load_k = [&](int j, uint4 (&raw)[NL]) __attribute__((always_inline)) {
      const uint16_t *krow = pk_base + (size_t)min(j, nk - 1) * D + 8 * part;    // (beyond nk: the last one, masked below)
#pragma unroll
      for (int t = 0; t < NL; t++) raw[t] = *(const uint4 *)(krow + 32 * t);
    };
    uint4 next[NL];
    load_k(c, next);
    double qd[D / 4];
    const uint16_t *qrow = pool_q + ((size_t)bh * nq + i) * D + 8 * part;
#pragma unroll
    for (int t = 0; t < NL; t++) {
      const uint4 v = *(const uint4 *)(qrow + 32 * t);
      const uint32_t w[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
      for (int e = 0; e < 8; e++) qd[8 * t + e] = (double)elem_to_f32<DT>((uint16_t)((e & 1) ? (w[e >> 1] >> 16) : (w[e >> 1] & 0xffffu)));
    }
#pragma unroll 1
    for (int j = c; j < NKP; j += COLS) {
      if (j - c >= causal_lim) {                        // uniform: no live column in this trip
        if (part == 0) s_score[j] = NEG_INF;
        continue;
      }
      uint4 kv[NL];
#pragma unroll
      for (int t = 0; t < NL; t++) kv[t] = next[t];
      load_k(j + COLS, next);
      const bool dead = j >= causal_lim || simk[min(j, nk - 1)] == 0;
      double acc = 0.0;
#pragma unroll
      for (int t = 0; t < NL; t++) {
        const uint32_t w[4] = {kv[t].x, kv[t].y, kv[t].z, kv[t].w};
#pragma unroll
        for (int e = 0; e < 8; e++)
          acc = __builtin_fma(qd[8 * t + e], (double)elem_to_f32<DT>((uint16_t)((e & 1) ? (w[e >> 1] >> 16) : (w[e >> 1] & 0xffffu))), acc);
      }
      acc = group_sum_f64<4>(acc);
      const float a1 = elem_to_f32<DT>(f64_to_elem_fast<DT>(acc));
      const uint16_t a2 = f64_to_elem_fast<DT>((double)a1 * (double)sm_scale);
      if (part == 0) s_score[j] = dead ? NEG_INF : a2;
    }
  }
  if (tid < 64) s_lsum[tid] = 0.0;
  __syncthreads();

  // ---- exponentials: wavefront w holds columns 64 (w + NW p) + lane; the maximum is taken by every wavefront for itself
  float lmax = -INFINITY;
#pragma unroll
  for (int t = 0; t < EPL; t++) lmax = fmaxf(lmax, elem_to_f32<DT>(s_score[64 * t + lane]));
  const float mx = wave_max_f32(lmax);
  double ev[P];
#pragma unroll
  for (int p = 0; p < P; p++) {
    const int j = 64 * (wave + NW * p) + lane;
    const float sc = elem_to_f32<DT>(s_score[j]);
    ev[p] = (sc == -INFINITY) ? 0.0 : cexp((double)sc - (double)mx);
    s_ev[j] = ev[p];
  }
  __syncthreads();
  // the fixed summation tree: lane l adds e[l], e[l+64], ... in order, then an xor butterfly (32 .. 1)
  double part = 0.0;
#pragma unroll
  for (int t = 0; t < EPL; t++) part = part + s_ev[64 * t + lane];
  const double total = wave_tree_sum_f64(part);

  // ---- probabilities -> sortable keys (the comment on the kernel above says why the product will do)
  const double rtotal = total > 0.0 ? 1.0 / total : 0.0;
  uint32_t okey[P], key[P];
#pragma unroll
  for (int p = 0; p < P; p++) {
    const int j = 64 * (wave + NW * p) + lane;
    okey[p] = j < nk ? ((probability_bits<DT>(ev[p], total, rtotal) << 16) | (0xffffu - (uint32_t)j)) : 0u;
    key[p] = okey[p];
  }
  long long n;
  uint32_t kth = 0u;
  if (by_topk) {
#pragma unroll
    for (int p = 0; p < P; p++) s_run[64 * (wave + NW * p) + lane] = okey[p];
    __syncthreads();
    const float t = level.at(h) * (float)nk;            // binary32 product, truncated (utils.py:405)
    n = (long long)t;
    if (n <= 0) n = 1;                                  // utils.py:289
    if (n < nk) {
      uint32_t all[EPL];
#pragma unroll
      for (int t2 = 0; t2 < EPL; t2++) all[t2] = s_run[64 * t2 + lane];
      kth = nth_largest_key<EPL>(all, (int)n);
    }
  } else {
    bitonic_sort_desc<P, 2>(key, lane);                 // sorted position of key[p] is lane * P + p
    uint32_t *run_w = s_run + RUN * wave;
#pragma unroll
    for (int p = 0; p < P; p++) run_w[lane * P + p] = key[p];
    for (int x = tid; x < NKP; x += NT)                 // the keys fill the first nk places
      if (x >= nk) s_sorted[x] = 0u;
    __syncthreads();
    // place of a key: its own in its run, plus the larger ones of every other run (keys below nk are distinct)
    int pos[P];
#pragma unroll
    for (int p = 0; p < P; p++) pos[p] = lane * P + p;
#pragma unroll
    for (int o = 1; o < NW; o++) {
      const uint32_t *r = s_run + RUN * ((wave + o) & (NW - 1));
#pragma unroll
      for (int p = 0; p < P; p++) {
        int cnt = 0;
#pragma unroll
        for (int s = RUN / 2; s >= 1; s >>= 1) cnt += r[cnt + s - 1] > key[p] ? s : 0;
        pos[p] += cnt + (r[cnt] > key[p] ? 1 : 0);      // cnt <= RUN - 1 here
      }
    }
#pragma unroll
    for (int p = 0; p < P; p++)
      if (key[p] != 0u) s_sorted[pos[p]] = key[p];
    __syncthreads();
    if (wave == 0) {
      uint32_t sk[EPL];
#pragma unroll
      for (int t = 0; t < EPL; t++) sk[t] = s_sorted[lane * EPL + t];
      // cdf[v] = T(sum_{u<=v} p_sorted[u]);  n = #{v < nk : cdf[v] <= threshold}  (utils.py:398-403)
      double lsum = 0.0;
#pragma unroll
      for (int t = 0; t < EPL; t++) lsum += (double)elem_to_f32<DT>((uint16_t)(sk[t] >> 16));
      s_lsum[64 + lane] = lsum;
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      __builtin_amdgcn_wave_barrier();
      // the sums of the lanes before this one, in their order: the window of 64 that ends there, zeros first
      double run = 0.0;
#pragma unroll 16
      for (int u = 0; u < 64; u++) run += s_lsum[lane + u];
      const double thr = (double)level.at(h);
      int cnt = 0;
#pragma unroll
      for (int t = 0; t < EPL; t++) {
        run += (double)elem_to_f32<DT>((uint16_t)(sk[t] >> 16));
        const float cdfv = elem_to_f32<DT>(f64_to_elem_fast<DT>(run));
        cnt += __builtin_popcountll(__ballot(lane * EPL + t < nk && (double)cdfv <= thr));
      }
      if (cnt <= 0) cnt = 1;                            // utils.py:289
      if (lane == 0) s_kth = cnt < nk ? s_sorted[cnt - 1] : 0u;
    }
    __syncthreads();
    kth = s_kth;
  }

  // ---- block map row, delta LUT: a kept column's place is the number of kept ones before it, its step the distance to the last of them
  const bool row_forced = sim_q[(size_t)bh * nq + i] == 0;
  const size_t row_off = ((size_t)bh * nq + i) * nk;
  uint64_t mine[P];
#pragma unroll
  for (int p = 0; p < P; p++) {
    const int j = 64 * (wave + NW * p) + lane;
    bool f = false;
    if (j < nk) {
      f = row_forced || (okey[p] >= kth) || (simk[j] == 0);
      if (j >= causal_lim) f = false;
      if (sink && j == 0) f = true;
      if (bmap != nullptr) bmap[row_off + j] = f ? 1 : 0;
    }
    mine[p] = __ballot(f);
    if (lane == 0) s_map[wave + NW * p] = mine[p];
  }
  __syncthreads();
  int base = 0, last = 0;                               // kept columns so far, the last of them
#pragma unroll
  for (int t = 0; t < EPL; t++) {
    const uint64_t m = s_map[t];
    if ((t & (NW - 1)) == wave) {                       // columns of this wavefront
      const uint64_t below = m & ((1ull << lane) - 1ull);
      if ((m >> lane) & 1ull)
        lut[row_off + base + __builtin_popcountll(below)] = 64 * t + lane - (below ? 64 * t + 63 - __builtin_clzll(below) : last);
    }
    base += __builtin_popcountll(m);
    if (m) last = 64 * t + 63 - __builtin_clzll(m);
  }
  for (int x = tid; x < nk; x += NT)
    if (x >= base) lut[row_off + x] = 0;
  if (tid == 0) {
    valid[(size_t)bh * nq + i] = base;
    if (valid_out != nullptr) valid_out[(size_t)bh * nq + i] = base;
  }
}

// =============================================================================================
// user mask -> LUT
// =============================================================================================
template <int KIND>
__global__ __launch_bounds__(256) void map_to_lut_kernel(const void *__restrict__ mask, int32_t *__restrict__ lut,
                                                         int32_t *__restrict__ valid, int nq, int nk, int nkp) {
  extern __shared__ __align__(16) unsigned char smem[];
  map_to_lut_body<KIND>(mask, lut, valid, nk, nkp, (size_t)blockIdx.y * nq + blockIdx.x, smem);
}

// =============================================================================================
// host launchers
// =============================================================================================
static int next_pow2_ge(int v, int lo) {
  int p = lo;
  while (p < v) p <<= 1;
  return p;
}

static int km_chunks(int B, int H, int N) {
  // enough workgroups to fill 256 CUs several times over, at least 256 rows each
  int want = (4096 + B * H - 1) / (B * H);
  int maxc = (N + 255) / 256;
  int c = want < maxc ? want : maxc;
  return c < 1 ? 1 : c;
}

size_t km_mean_workspace_bytes(int B, int H, int N, int D) {
  return (size_t)B * H * km_chunks(B, H, N) * D * sizeof(double);
}

template <int D, int DT>
static void launch_km(const void *k, Strides ks, void *km, void *ws, int B, int H, int N, hipStream_t st) {
  const int nchunk = km_chunks(B, H, N);
  const int rpc = (N + nchunk - 1) / nchunk;
  km_partial_kernel<D, DT><<<dim3(nchunk, B * H), 256, 0, st>>>((const uint16_t *)k, ks, H, (double *)ws, N, rpc);
  km_final_kernel<DT><<<B * H, dim3(D, 8), 0, st>>>((const double *)ws, (uint16_t *)km, nchunk, D, N);
}

void launch_km_mean(const void *k, Strides ks, void *km, void *ws, int B, int H, int N, int D, int dtype, hipStream_t st) {
  if (D == 64) { if (dtype == 0) launch_km<64, 0>(k, ks, km, ws, B, H, N, st); else launch_km<64, 1>(k, ks, km, ws, B, H, N, st); }
  else         { if (dtype == 0) launch_km<128, 0>(k, ks, km, ws, B, H, N, st); else launch_km<128, 1>(k, ks, km, ws, B, H, N, st); }
}

// ---- K column mean without a caller-provided workspace ---------------------------------------------------------
// The per-chunk partial sums go to a fixed array in device memory that the library owns (one copy per GPU, alive
// until the process ends).  In host code the array's NAME is only a handle: its device address is asked for once per
// device with hipGetSymbolAddress and that pointer is what the kernels receive.  Every call on a GPU shares the
// array, so two calls that overlap in time on one GPU (different streams or threads) race; calls on one stream are
// ordered.  Nothing needs clearing between calls: km_partial writes every partial sum km_final reads.
static __device__ __align__(256) unsigned char km_static_scratch[SPG_KM_STATIC_SCRATCH_BYTES];

size_t km_mean_static_capacity() { return SPG_KM_STATIC_SCRATCH_BYTES; }

hipError_t launch_km_mean_static(const void *k, Strides ks, void *km, int B, int H, int N, int D, int dtype, hipStream_t st) {
  constexpr int MAX_DEV = 64;
  static std::atomic<void *> scratch_of_device[MAX_DEV];
  int dev = -1;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return e;
  if (dev < 0 || dev >= MAX_DEV) return hipErrorInvalidDevice;
  // The array's address is looked up for, and only valid on, the CURRENT device: a stream that belongs to another GPU
  // would run the kernels there with this GPU's address.  (The null stream always belongs to the current device.)
  if (st != nullptr) {
    hipDevice_t sdev = -1;
    e = hipStreamGetDevice(st, &sdev);
    if (e != hipSuccess) return e;
    if ((int)sdev != dev) return hipErrorInvalidDevice;
  }
  void *ptr = scratch_of_device[dev].load(std::memory_order_acquire);
  if (ptr == nullptr) {
    // first call on this device (the device is current): resolve this GPU's copy of the array
    e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(km_static_scratch));
    if (e != hipSuccess) return e;
    if (ptr == nullptr) return hipErrorInvalidSymbol;
    scratch_of_device[dev].store(ptr, std::memory_order_release);
  }
  launch_km_mean(k, ks, km, ptr, B, H, N, D, dtype, st);
  return hipSuccess;
}

template <int BS, int D, int DT>
static void launch_psq3(const void *x, Strides xs, const void *km, void *pool, uint8_t *sim, int8_t *xq, float *scale,
                        const float *thr, int B, int H, int N, int quant_rows, hipStream_t st) {
  const int nb = (N + BS - 1) / BS;
  const dim3 grid((N + 127) / 128, B * H);      // one workgroup per 128 rows: one or two blocks
  const uint16_t *xp = (const uint16_t *)x, *kp = (const uint16_t *)km;
  uint16_t *pp = (uint16_t *)pool;
  if constexpr (BS == 128) {
    if (quant_rows == 32) {                     // per-warp granularity of Q (no mean: the C ABI refuses the combination)
      if (pool != nullptr) pool_sim_quant_kernel<BS, D, DT, false, true, 32><<<grid, 256, 0, st>>>(xp, xs, kp, pp, sim, xq, scale, thr, H, N, nb);
      else                 pool_sim_quant_kernel<BS, D, DT, false, false, 32><<<grid, 256, 0, st>>>(xp, xs, kp, pp, sim, xq, scale, thr, H, N, nb);
      return;
    }
  }
  if (pool != nullptr) {
    if (km) pool_sim_quant_kernel<BS, D, DT, true, true><<<grid, 256, 0, st>>>(xp, xs, kp, pp, sim, xq, scale, thr, H, N, nb);
    else    pool_sim_quant_kernel<BS, D, DT, false, true><<<grid, 256, 0, st>>>(xp, xs, kp, pp, sim, xq, scale, thr, H, N, nb);
  } else {
    if (km) pool_sim_quant_kernel<BS, D, DT, true, false><<<grid, 256, 0, st>>>(xp, xs, kp, pp, sim, xq, scale, thr, H, N, nb);
    else    pool_sim_quant_kernel<BS, D, DT, false, false><<<grid, 256, 0, st>>>(xp, xs, kp, pp, sim, xq, scale, thr, H, N, nb);
  }
}

void launch_pool_sim_quant(const void *x, Strides xs, const void *km, void *pool, uint8_t *sim, int8_t *xq, float *scale,
                           const float *thr, int B, int H, int N, int D, int block, int quant_rows, int dtype,
                           hipStream_t st) {
#define SPG_PSQ(BS_, D_, DT_) launch_psq3<BS_, D_, DT_>(x, xs, km, pool, sim, xq, scale, thr, B, H, N, quant_rows, st)
  if (block == 128) {
    if (D == 64) { if (dtype == 0) SPG_PSQ(128, 64, 0); else SPG_PSQ(128, 64, 1); }
    else         { if (dtype == 0) SPG_PSQ(128, 128, 0); else SPG_PSQ(128, 128, 1); }
  } else {
    if (D == 64) { if (dtype == 0) SPG_PSQ(64, 64, 0); else SPG_PSQ(64, 64, 1); }
    else         { if (dtype == 0) SPG_PSQ(64, 128, 0); else SPG_PSQ(64, 128, 1); }
  }
#undef SPG_PSQ
}

int block_select_max_nk() { return 8192; }

// Kernels that need more than 48 KiB of dynamic LDS must be told so once (per device); the size granted last is
// remembered per kernel and device, so the attribute call is not repeated on every launch.  gfx950 has 160 KiB of LDS
// per workgroup; a request beyond it (including the kernel's static arrays, at most 4 KiB here) is refused up front.
template <auto Kern>
static hipError_t allow_dynamic_lds(size_t lds) {
  if (lds + 4096 > 160 * 1024) return hipErrorInvalidConfiguration;
  if (lds <= 48 * 1024) return hipSuccess;
  static std::atomic<size_t> granted[32];
  int dev = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return e;
  const bool tracked = dev >= 0 && dev < 32;
  if (tracked && granted[dev].load(std::memory_order_relaxed) >= lds) return hipSuccess;
  e = hipFuncSetAttribute((const void *)Kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
  if (e == hipSuccess && tracked) granted[dev].store(lds, std::memory_order_relaxed);
  return e;
}

void launch_div_selftest(unsigned long long *counts, int n_div, uint32_t seed, hipStream_t st) {
  div_selftest_kernel<<<(n_div + 255) / 256, 256, 0, st>>>(counts, n_div, seed);
}

template <int D, int DT, int R>
static hipError_t launch_bs3(const void *pq, const uint8_t *sq, const void *pk, const uint8_t *sk, bool by_topk,
                             Hyper level, int causal, int sink, int32_t *lut, int32_t *valid, int32_t *valid_out, uint8_t *bmap, int B,
                             int H, int Hkv, int nq, int nk, int nkp, hipStream_t st) {
  const size_t lds = (size_t)R * D * 8 + (size_t)R * nkp * 4 + 12 * (size_t)nkp;
  auto kern = block_select_kernel<D, DT, R>;
  {
    hipError_t e = allow_dynamic_lds<block_select_kernel<D, DT, R>>(lds);
    if (e != hipSuccess) return e;
  }
  kern<<<dim3((nq + R - 1) / R, B * H), 256, lds, st>>>((const uint16_t *)pq, sq, (const uint16_t *)pk, sk, by_topk, level,
                                                        causal, sink, lut, valid, valid_out, bmap, H, Hkv, nq, nk, nkp);
  return hipSuccess;
}

template <int D, int DT>
static hipError_t launch_bs2(const void *pq, const uint8_t *sq, const void *pk, const uint8_t *sk, bool by_topk,
                             Hyper level, int causal, int sink, int32_t *lut, int32_t *valid, int32_t *valid_out, uint8_t *bmap, int B,
                             int H, int Hkv, int nq, int nk, hipStream_t st) {
  const int nkp = next_pow2_ge(nk, 256);
  if (nkp <= 2048) {
    // a whole row fits the registers of one wavefront
    // A workgroup to a row where two of them per CU hold all rows; a whole call in us with the kernels below / with this (top-k 0.05,
    // D=64): 256 rows nk 256 37.5 / 34.3, nk 512 57.2 / 49.8, nk 1875 145.1 / 118.9; 512 rows nk 141 44.5 / 42.8, nk 278 60.7 / 58.8, nk 1875
    // 217.1 / 199.3; CDF, D=128: 64 rows nk 141 69.5 / 64.8, 512 rows nk 278 317.1 / 312.6.  With 640 rows it is down to +-1 %, with
    // 1112 rows nk 278 (top-k, D=128) 321.6 / 334.2: a wavefront to a row does less in all.
    if ((long long)nq * B * H <= 512) {
#define SPG_BSR(EPL_)                                                                                                        \
      block_select_row_kernel<D, DT, EPL_><<<dim3(nq, B * H), EPL_ == 4 ? 256 : 512, 0, st>>>(                               \
          (const uint16_t *)pq, sq, (const uint16_t *)pk, sk, by_topk, level, causal, sink, lut, valid, valid_out, bmap, H, Hkv, nq, nk)
      if (nkp == 256) SPG_BSR(4);
      else if (nkp == 512) SPG_BSR(8);
      else if (nkp == 1024) SPG_BSR(16);
      else SPG_BSR(32);
#undef SPG_BSR
      return hipSuccess;
    }
#define SPG_BSW(NW_, EPL_, DUAL_, R_)                                                                                    \
    {                                                                                                           \
      const size_t lds = (size_t)R_ * nkp * 2 + (size_t)NW_ * nkp * 2 + NW_ * 64 * 8;                           \
      auto kern = block_select_wave_kernel<D, DT, NW_, EPL_, DUAL_, R_>;                                                   \
      {                                                                                                         \
        hipError_t e = allow_dynamic_lds<block_select_wave_kernel<D, DT, NW_, EPL_, DUAL_, R_>>(lds);                      \
        if (e != hipSuccess) return e;                                                                          \
      }                                                                                                         \
      kern<<<dim3((nq + R_ - 1) / R_, B * H), 64 * NW_, lds, st>>>((const uint16_t *)pq, sq, (const uint16_t *)pk, sk, by_topk, \
                                                               level, causal, sink, lut, valid, valid_out, bmap, H, Hkv, nq, nk); \
      return hipSuccess;                                                                                        \
    }
    // Eight rows instead of sixteen per workgroup, one per wavefront, where sixteen leave a CU with little more than one
    // workgroup: the time is then that of one wavefront's rows, and the half-empty score tiles cost less than the second row.
    // us with 16 / 8: 96 workgroups D=128 nk=128 15.3 / 10.4, 128 D=128 nk=256 25.4 / 16.9, 192 D=64 nk=256 21.5 / 18.2, 270 D=64
    // nk=278 44.0 / 35.7, 49 D=128 nk=1563 130 / 85; 512 D=128 nk=512 46.6 / 64.1.
    const bool few = (nq + 15) / 16 * B * H <= (D == 64 ? 384 : 256);
    if (nkp == 256) { if (few) SPG_BSW(8, 4, false, 8) else SPG_BSW(8, 4, false, 16) }
    if (nkp == 512) { if (few) SPG_BSW(8, 8, false, 8) else SPG_BSW(8, 8, false, 16) }
    if (nkp == 1024) { if (few) SPG_BSW(8, 16, false, 8) else SPG_BSW(8, 16, false, 16) }
    if (few) SPG_BSW(8, 32, true, 8) else SPG_BSW(8, 32, true, 16)
#undef SPG_BSW
  }
  // rows per workgroup: reuse of the pooled-K reads against LDS footprint (scores are R*nkp floats)
  if (nkp <= 1024) return launch_bs3<D, DT, 8>(pq, sq, pk, sk, by_topk, level, causal, sink, lut, valid, valid_out, bmap, B, H, Hkv, nq, nk, nkp, st);
  if (nkp <= 4096) return launch_bs3<D, DT, 4>(pq, sq, pk, sk, by_topk, level, causal, sink, lut, valid, valid_out, bmap, B, H, Hkv, nq, nk, nkp, st);
  // nkp = 8192: one row per workgroup (D*8 + 16*nkp = 129 KiB; two rows would need 162 KiB, more than the 160 KiB a
  // workgroup can have)
  return launch_bs3<D, DT, 1>(pq, sq, pk, sk, by_topk, level, causal, sink, lut, valid, valid_out, bmap, B, H, Hkv, nq, nk, nkp, st);
}

hipError_t launch_block_select_h(const void *pq, const uint8_t *sq, const void *pk, const uint8_t *sk, bool by_topk,
                                 Hyper level, int causal, int sink, int32_t *lut, int32_t *valid, int32_t *valid_out, uint8_t *bmap,
                                 int B, int H, int Hkv, int nq, int nk, int D, int dtype, hipStream_t st) {
#define SPG_BS(D_, DT_) return launch_bs2<D_, DT_>(pq, sq, pk, sk, by_topk, level, causal, sink, lut, valid, valid_out, bmap, B, H, Hkv, nq, nk, st)
  if (D == 64) { if (dtype == 0) SPG_BS(64, 0); else SPG_BS(64, 1); }
  else         { if (dtype == 0) SPG_BS(128, 0); else SPG_BS(128, 1); }
#undef SPG_BS
}

hipError_t launch_block_select(const void *pq, const uint8_t *sq, const void *pk, const uint8_t *sk, const float *topk,
                               const float *cdf, int causal, int sink, int32_t *lut, int32_t *valid, uint8_t *bmap,
                               int B, int H, int Hkv, int nq, int nk, int D, int dtype, hipStream_t st) {
  return launch_block_select_h(pq, sq, pk, sk, topk != nullptr, Hyper{topk != nullptr ? topk : cdf, 0.f}, causal, sink, lut, valid,
                               nullptr, bmap, B, H, Hkv, nq, nk, D, dtype, st);
}

hipError_t launch_map_to_lut(const void *mask, int kind, int32_t *lut, int32_t *valid, int B, int H, int nq, int nk,
                             hipStream_t st) {
  const int nkp = next_pow2_ge(nk, 256);
  const size_t lds = 4 * (size_t)nkp + 64;
  const dim3 grid(nq, B * H);
#define SPG_M2L(K_)                                                                                      \
  case K_: {                                                                                             \
    auto kern = map_to_lut_kernel<K_>;                                                                   \
    {                                                                                                    \
      hipError_t e = allow_dynamic_lds<map_to_lut_kernel<K_>>(lds);                                      \
      if (e != hipSuccess) return e;                                                                     \
    }                                                                                                    \
    kern<<<grid, 256, lds, st>>>(mask, lut, valid, nq, nk, nkp);                                         \
    break;                                                                                               \
  }
  switch (kind) {
    SPG_M2L(0) SPG_M2L(1) SPG_M2L(2) SPG_M2L(3) SPG_M2L(4) SPG_M2L(5) SPG_M2L(6)
    default: return hipErrorInvalidValue;
  }
#undef SPG_M2L
  return hipSuccess;
}

}  // namespace spg
