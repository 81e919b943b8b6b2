// Block-sparse INT8-QK / FP8-PV attention for gfx950 (CDNA4), written for 64-lane wavefronts and MFMA.
//
// Replaces qk_int_sv_f8_block_sparse_attn_kernel (csrc/qattn/qk_int_sv_f8_cuda_sm89.cuh:42-755) as launched by
// qk_int8_sv_f8_accum_f32_block_sparse_attn_inst_buf_fuse_v_scale_with_pv_threshold
// (csrc/qattn/qk_int_sv_f8_cuda_sm89.cu:197-390): per-block or per-warp INT8 scales (qk_quant_gran 1 / 2), PV threshold
// per block (or per 32 rows, or none), fp32 PV accumulation, V scale fused into the epilogue.
//
// Design (not a translation of the mma.sync tiling):
//  * one workgroup = one 128-row Q block = 4 wavefronts x 32 queries;
//  * both products are computed TRANSPOSED so that a lane owns one query column throughout:
//        S^T (64 keys x 32 queries) = K . Q^T   v_mfma_i32_32x32x32_i8     (A = K rows from LDS, B = Q in VGPRs)
//        O^T (D x 32 queries)      += V^T . P^T v_mfma_f32_32x32x64_f8f6f4 (A = V^T rows from LDS, B = P in VGPRs)
//    lane l holds query l%32; lanes l and l^32 hold the two halves of that query's keys / output channels.
//    Row max / row sum are lane-local plus ONE cross-lane exchange; the O rescale is lane-local.
//  * the K rows are assigned to MFMA rows through a permutation chosen such that, after S^T is computed, the
//    32 scores a lane holds belong to 32 CONSECUTIVE keys (32*half .. 32*half+31): packing them to e4m3 gives the
//    B operand of the PV MFMA with no shuffle, and the matching A operand is 32 contiguous bytes of a V^T row;
//  * V lives in HBM as [nk][D][64] e4m3 tiles (one contiguous 64*D-byte read per block), K as (N,D) int8 rows;
//  * K/V tiles go HBM/L2 -> LDS directly (global_load_lds_dwordx4, no VGPR staging) through a 3-deep LDS ring:
//    the tiles of block it+2 are in flight while block it is computed, and ONE workgroup barrier per block covers
//    both the tile hand-over and the workgroup-wide PV-skip vote (the FP16-PV variant, whose V^T tiles are twice as
//    large, uses two-slot rings so that three workgroups still share a CU);
//  * the INT8 scale of Q is read per 128-row block or per wavefront of 32 rows (qk_quant_gran 1 / 2): a wavefront IS
//    the 32-row group, so the scale stays a scalar either way;
//  * LDS tiles are unpadded; bank conflicts are avoided by an XOR swizzle of the 16-byte chunks inside a row
//    (applied to the per-lane global address for K, baked into the HBM tile layout for V);
//  * the INT8 accumulators start at the bit pattern of the float 1/(2 pi), an inline constant of the instruction set (no
//    register or LDS read initialises them): read as a float the int32 result is 1/(2 pi) + dot * 2^-26, so the scores need
//    no int-to-float conversion; the constant is folded into the additive term of the fma that feeds exp2;
//  * only "skip" votes of the PV threshold reach LDS, and the rescale factor of O is computed only in iterations in which
//    a running maximum rose;
//  * workgroup ids are remapped so that one XCD (one L2) works on one head at a time, heaviest rows first;
//  * on large grids at D = 128 a workgroup quantises its own Q block before it starts (FQ; q_in_front has the line and the figures).
#include "common.h"
#include "launch.h"
#include "lds_asm.h"
#include "select_row.h"
#include "stage_bodies.h"

#include <type_traits>

namespace spg {

typedef int v8i __attribute__((ext_vector_type(8)));
typedef int v8i_a16 __attribute__((ext_vector_type(8), aligned(16)));
typedef int v16i __attribute__((ext_vector_type(16)));
typedef float v16f __attribute__((ext_vector_type(16)));

// Results of psq_core for one Q block in LDS.  A code row of D bytes has its 16-byte chunks at chunk ^ swz(row): the Q operand is read by 32
// lanes of as many rows, which spreads them over the sixteen slots of a 256-byte line.
template <int D>
struct PsqToLds {
  static constexpr bool ALL_ROWS = true;
  uint16_t *pool_at;
  uint32_t *sim_at;
  float *scale_at;
  unsigned char *lo, *hi;             // rows 0-63 and 64-127
  bool one;
  static_assert(D == 128, "two rows to a line");
  static __device__ __forceinline__ int swz(int row) { return (row >> 1) & 7; }
  __device__ __forceinline__ bool one_scale() const { return one; }
  __device__ __forceinline__ void pool(int, int col, uint16_t v) const { pool_at[col] = v; }
  __device__ __forceinline__ void sim(int, bool v) const { *sim_at = v ? 1 : 0; }
  __device__ __forceinline__ void codes(int row, int c, uint2 v) const {
    *(uint2 *)((row < 64 ? lo : hi) + (row & 63) * D + ((c >> 1) ^ swz(row)) * 16 + (c & 1) * 8) = v;
  }
  __device__ __forceinline__ void scale(int g, float v) const { scale_at[g] = v; }
};

#define SPG_NEG_BIG (-5000000.0f)   // csrc/qattn/attn_utils.cuh:350, qk_int_sv_f8_cuda_sm89.cuh:171
#define SPG_FP8_OFFSET 8.807f       // csrc/qattn/attn_utils.cuh:28
#define SPG_ACC_C_BITS 0x3E22F983    // the float 1/(2 pi), an inline constant of the instruction set: initial accumulator
#define SPG_ACC_SCALE 67108864.0f    // 2^26: one unit of the integer dot product is 2^-26 in the binade [1/8, 1/4)
#define SPG_ROW_MAJOR_MAX 512       // workgroups per XCD up to which causal rows are ordered by length across heads
#define SPG_QUEUE_MIN 384           // workgroups per XCD (four rounds of 32 CUs x 3) and ...
#define SPG_QUEUE_MIN_ROW 16384     // ... length of a row, in channels of K blocks, beyond which the queue pays (launch_attn)
#define SPG_QUEUE_EXTRA 12          // one workgroup in so many is launched on top
#define SPG_PLACES 96               // last rows of an XCD that lower their priority: 32 CUs x 3, the rows it works on at a time at D = 128.  D = 64
                                    // fits four workgroups per CU (124 registers, 25 KB): 112 and 128 make no difference there, one number for both
#define SPG_START_PRIO_MAX 1024     // workgroups, beyond the places for them, up to which rows that select in place start at the loop's priority
#define SPG_LOG2E 1.44269504088896340736f

// n / d for 0 <= n < 2^31 as a multiplication and a shift: m = ceil(2^(31+s) / d) with 2^(s-1) < d <= 2^s is a 32-bit number, and
// m d - 2^(31+s) < d <= 2^s keeps the truncated product exact.  (A division by a launch argument is some 40 dependent
// instructions; a workgroup needs six of them before it can ask for its data.)
struct FastDiv {
  uint32_t m, s;
  static FastDiv of(int d) {
    FastDiv f = {0, 0};
    while ((1ll << f.s) < d) f.s++;
    f.m = (uint32_t)(((1ull << (31 + f.s)) + (unsigned)d - 1) / (unsigned)d);
    return f;
  }
  __device__ __forceinline__ int operator()(int n) const { return (int)(__umulhi((uint32_t)n << 1, m) >> s); }
};

struct AttnParams {
  const int8_t *q8, *k8;
  const uint8_t *v8;
  void *out;
  Strides os;      // element strides of out (B, H, N, D), last dimension contiguous
  const int32_t *lut, *valid;
  Hyper pvthr;
  const float *q_scale, *k_scale, *v_scale;
  int32_t *pv_count;
  int B, H, Hkv, N, Nk, nq, nk;   // N query rows, Nk key/value rows per head (qo_len / kv_len of sm89.cu:256-300)
  float sm_scale_log2;
  int is_causal;
  int pv_mode;     // PVThresholdMode of the reference (attn_utils.cuh:58-62): 0 none, 1 per block, 2 per wavefront of 32 rows
  int q_per_warp;  // QuantGranularity of Q (sm89.cuh:106-121): 0 one scale per 128-row block, 1 one per 32 rows (B,H,nq*4)
  int total_wg, wg_per_xcd;
  int *queue;      // NULL, or 8 counters, zero at the start (take_item)
  FastDiv by_nq, by_rest, by_H, by_group;   // nq, nq - rows_first, H, H / Hkv
  int rows_first;  // so many of the longest rows of every head come before the rest (place_workgroup)
  RowSelect sel;   // selection inside the kernel (template argument SEL); lut is unused then
  RawQ q;          // Q as the caller has it (template argument FQ); q8, q_scale, sel.pool_q and sel.sim_q are unused then
  int few;         // workgroups to a row (few_rows_attn_kernel), or 0
  RowSplit split;  // rows in chunks (template argument SPLIT)
  FastDiv by_chunks;    // (rows + 7) / 8 (place_part)
};

// The chunks of a row with `nv` blocks: as few as hold at most `split.per` of them each, of equal length; chunk c is places begin(c) to
// begin(c + 1) - 1 of the list.  A row's last two blocks are in its last chunk.
struct RowChunks {
  uint32_t nv, n;
  __device__ __forceinline__ RowChunks(int nv_, const RowSplit &split)
      : nv((uint32_t)nv_), n((uint32_t)max(1, min(split.chunks, (nv_ + split.per - 1) / split.per))) {}
  __device__ __forceinline__ int begin(int c) const { return (int)((uint32_t)c * nv / n); }
  // Rows start at different chunks: workgroups that start together would else ask for the same tiles at the same time.  us per call, one
  // head N17776, all rows from their first / in turn: D64 top-k 0.5 100.3 / 96.6, all blocks kept 139.8 / 135.0; D128 2 x 14000 145.0 / 141.9.
  __device__ __forceinline__ int turned(int part, int row) const { return (int)((uint32_t)(part + row) % n); }
};
// Workgroup -> (row, part of it).  An XCD works on consecutive rows of a head, from the last one down; the first parts of all its rows
// come first, so that parts which shorter rows do not have leave no gaps among those that are there.
__device__ __forceinline__ bool place_part(const AttnParams &p, int id, int &bh, int &qb, int &part) {
  const int x = id & 7, j = id >> 3, first = x * p.split.rows >> 3, rows = ((x + 1) * p.split.rows >> 3) - first;
  part = p.by_chunks(j);
  const int i = j - part * ((p.split.rows + 7) >> 3);
  if (i >= rows) return false;
  bh = p.by_nq(first + i);
  qb = p.nq - 1 - (first + i - bh * p.nq);
  return true;
}
// inclusive prefix sums over a wavefront (DPP: shifts within rows of sixteen, then the last lane of a row to those behind it)
__device__ __forceinline__ int wave_prefix_sum(int v) {
  v += __builtin_amdgcn_update_dpp(0, v, 0x111, 0xf, 0xf, false);
  v += __builtin_amdgcn_update_dpp(0, v, 0x112, 0xf, 0xf, false);
  v += __builtin_amdgcn_update_dpp(0, v, 0x114, 0xf, 0xf, false);
  v += __builtin_amdgcn_update_dpp(0, v, 0x118, 0xf, 0xf, false);
  v += __builtin_amdgcn_update_dpp(0, v, 0x142, 0xa, 0xf, false);
  v += __builtin_amdgcn_update_dpp(0, v, 0x143, 0xc, 0xf, false);
  return v;
}

// Workgroup -> (batch*head, q block).  Ids are dealt round-robin over the 8 XCDs; each XCD (one L2) gets a contiguous
// range of (head, row) pairs, rows from the last one down: causal rows get longer with the row index, and a partial last
// Q block is never "similar", so all its blocks are kept.
// Within the range the order is head by head, so that the resident workgroups share K/V tiles - except that the first
// `rows_first` rows of ALL heads of the range come first: a long row that starts when the rest of the chip is about to
// finish runs on alone.  (Measured with head-by-head order: H30 N17776 D64, whose partial last rows are twice as long as the
// others, last workgroup at 1150 us with the median CU done at 1034; causal H32 N4096, 101 us against 81.)
__device__ __forceinline__ bool place_workgroup(const AttnParams &p, int xcd, int j, int &bh, int &qb) {
  const int L0 = xcd * p.wg_per_xcd, L1 = min(L0 + p.wg_per_xcd, p.total_wg);
  if (L0 + j >= L1) return false;
  const int nq = p.nq, T = p.rows_first;
  // the range is rows a.. of head h0 (if a > 0), all rows of F heads from hf on, rows ..b-1 of head h1 (if b > 0)
  const int h0 = p.by_nq(L0), a = L0 - h0 * nq, h1 = p.by_nq(L1), b = L1 - h1 * nq;
  const int hf = h0 + (a > 0 ? 1 : 0), F = h1 - hf;
  int h, t;
  if (T == 0 || F < 0) {
    h = p.by_nq(L0 + j);
    t = L0 + j - h * nq;
  } else {
    auto upto = [&](int rows) { return F * rows + (a > 0 ? max(0, rows - a) : 0) + min(rows, b); };   // pairs with row < rows
    if (j < upto(T)) {
      int lo = 0, hi = T - 1;                        // largest row with upto(row) <= j
      while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (upto(mid) <= j) lo = mid; else hi = mid - 1;
      }
      t = lo;
      int i = j - upto(t);
      const int first = a > 0 && t >= a ? 1 : 0;
      h = i < first ? h0 : hf + (i - first);         // the partial last head h1 = hf + F follows the full ones
    } else {
      j -= upto(T);
      const int n0 = a > 0 ? nq - max(a, T) : 0, per = nq - T;
      if (j < n0) { h = h0; t = max(a, T) + j; }
      else {
        j -= n0;
        const int i = per > 0 ? p.by_rest(j) : 0;
        h = hf + min(i, F);
        t = T + j - min(i, F) * per;
      }
    }
  }
  bh = h;
  qb = nq - 1 - t;
  return true;
}

// With a queue the j-th place of a range goes to whoever asks for it next, and a workgroup whose own XCD has nothing left
// asks the others: the XCDs do not run at one speed (the fastest and the slowest differ by 5 to 6 % in the time they take for
// equal shares of a long grid, the same ones on every launch), and a fixed share each leaves the fast ones idle at the end.
// The grid holds SPG_QUEUE_EXTRA more workgroups than places, so that a fast XCD is dealt enough of them; one that finds
// nothing ends.  Called by one thread.
__device__ __forceinline__ int take_item(const AttnParams &p, int w) {
  for (int i = 0; i < 8; i++) {
    const int x = (w + i) & 7;
    const int size = min(p.wg_per_xcd, p.total_wg - x * p.wg_per_xcd);
    const int j = size > 0 ? __hip_atomic_fetch_add(p.queue + x, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) : 0;
    if (j < size) return (j << 3) | x;
  }
  return -1;
}

// v_max_f32 as one instruction: fmaxf() on a value the compiler cannot prove to be a quiet number (a loop-carried
// maximum, the output of a lane exchange) costs a canonicalising self-maximum per operand first.  The operands here are
// products and maxima of finite numbers.
__device__ __forceinline__ float max_raw(float a, float b) {
  float r;
  asm("v_max_f32 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
  return r;
}
__device__ __forceinline__ float half_swap_max_raw(float v) {
  float lo, hi, r;
  half_swap(v, lo, hi);
  asm("s_nop 0\n\tv_max_f32 %0, %1, %2" : "=v"(r) : "v"(lo), "v"(hi));   // one idle state behind the lane exchange
  return r;
}
// e4m3 pack of the probabilities.  v_cvt_pk_fp8_f32 returns NaN (0x7f) for |x| > 464 unless MODE.FP16_OVFL is set, in
// which case finite values clamp to +-448 like the reference's cvt.rn.satfinite.e4m3x2.f32 (csrc/numeric_conversion.cuh:48-63);
// the bit is set once per wavefront, costs nothing per element and affects no other instruction this kernel depends on
// (the fp16 epilogue conversion cannot overflow: |O / d| <= max |V|).
__device__ __forceinline__ void fp8_saturation_on() {
  __builtin_amdgcn_s_setreg(1 | (23 << 6) | (0 << 11), 1);   // hwreg(HW_REG_MODE, offset 23, size 1) = FP16_OVFL
}
__device__ __forceinline__ int pack4_e4m3(float x0, float x1, float x2, float x3) {
  // both halves of the destination are written, so its initial content is irrelevant: start from a register that is
  // "defined" by an empty asm instead of a zeroed one
  int wv;
  asm volatile("" : "=v"(wv));
  wv = __builtin_amdgcn_cvt_pk_fp8_f32(x0, x1, wv, false);
  wv = __builtin_amdgcn_cvt_pk_fp8_f32(x2, x3, wv, true);
  return wv;
}

// Self test of the pack: codes[i] = e4m3(x[i]) exactly as the attention kernel produces it (saturate != 0) or as the bare
// instruction does (saturate == 0).  n is a multiple of 4.
__global__ __launch_bounds__(256) void fp8_pack_selftest_kernel(const float *__restrict__ x, uint32_t *__restrict__ codes,
                                                                int n4, int saturate) {
  if (saturate) fp8_saturation_on();
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i >= n4) return;
  const float4 v = ((const float4 *)x)[i];
  codes[i] = (uint32_t)pack4_e4m3(v.x, v.y, v.z, v.w);
}
void launch_fp8_pack_selftest(const float *x, uint8_t *codes, int n, int saturate, hipStream_t st) {
  const int n4 = n / 4;
  fp8_pack_selftest_kernel<<<(n4 + 255) / 256, 256, 0, st>>>(x, (uint32_t *)codes, n4, saturate);
}

// Output rows of one wavefront, O / d * v_scale rounded to the output type: through LDS (`orow_lds`, 32 rows) and out as whole rows,
// 16 bytes per lane.
constexpr int orow_bytes(int D) { return 2 * D + 16; }      // padded row: the 8-byte writes of 32 rows spread over the banks
template <int D, int ODT, bool PV16>
__device__ __forceinline__ void store_rows(const v16f (&O)[D / 32], float inv, unsigned char *orow_lds, const float *v_scale, const AttnParams &p,
                                           int batch, int head, int row0, uint32_t lane) {
  constexpr int NDT = D / 32, OROW = orow_bytes(D);
  const int r_e = (int)lane & 31, hh_e = (int)lane >> 5;
#pragma unroll
  for (int dt = 0; dt < NDT; dt++) {
#pragma unroll
    for (int g = 0; g < 4; g++) {
      const int d0 = 32 * dt + 8 * g + 4 * hh_e;
      float4 sc = make_float4(1.f, 1.f, 1.f, 1.f);
      if constexpr (!PV16) sc = *(const float4 *)(v_scale + d0);
      const uint16_t o0 = f32_to_elem<ODT>(O[dt][4 * g + 0] * inv * sc.x);
      const uint16_t o1 = f32_to_elem<ODT>(O[dt][4 * g + 1] * inv * sc.y);
      const uint16_t o2 = f32_to_elem<ODT>(O[dt][4 * g + 2] * inv * sc.z);
      const uint16_t o3 = f32_to_elem<ODT>(O[dt][4 * g + 3] * inv * sc.w);
      *(uint2 *)(orow_lds + r_e * OROW + d0 * 2) = make_uint2((uint32_t)o0 | ((uint32_t)o1 << 16), (uint32_t)o2 | ((uint32_t)o3 << 16));
    }
  }
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
  constexpr int LPR = D / 8, RPI = 64 / LPR;                 // lanes per row, rows per store instruction
  uint16_t *obase = (uint16_t *)p.out + (size_t)batch * p.os.sb + (size_t)head * p.os.sh + ((int)lane % LPR) * 8;
#pragma unroll
  for (int i = 0; i < 32 / RPI; i++) {
    const int row = i * RPI + (int)lane / LPR, grow = row0 + row;
    const uint4 t = *(const uint4 *)(orow_lds + row * OROW + ((int)lane % LPR) * 16);
    if (grow < p.N) *(uint4 *)(obase + (size_t)grow * p.os.sn) = t;
  }
}

// 16-byte-chunk swizzles.  K tile row = key (D bytes, D/16 chunks); V^T tile row = channel (64 bytes, 4 chunks).
// The LDS serves a ds_read_b128 one half-wavefront (32 lanes) at a time and needs two clocks for it when the 32
// addresses fall evenly on the sixteen 16-byte slots of a 256-byte line (two lanes per slot); a slot that is hit 2k
// times costs k times as much.  The slot of an address is (byte offset mod 256) / 16, so the low row bits already select
// part of it (one bit for 128-byte rows, two bits for 64-byte rows) and the swizzle must come from OTHER row bits that
// vary inside a half-wavefront: for the K operand lane r reads key row 32*((r>>2)&1) + 4*(r>>3) + (r&3) (+16 for the
// second tile), for the V^T operand lane r reads channel row r (+32 per output tile).
template <int D>
__device__ __forceinline__ uint32_t k_swz(uint32_t row) {
  if constexpr (D == 128) return ((row >> 1) & 3u) | (((row >> 5) & 1u) << 2);
  else return ((row >> 2) & 1u) | (((row >> 5) & 1u) << 1);
}
__device__ __forceinline__ int v_swz(int row) { return (row >> 2) & 3; }

// PV16 = false: V^T tiles are e4m3 (64 bytes per channel row), P is packed to e4m3 with the +8.807 exponent offset and
//               the denominator sums the un-rounded P (the SageAttention2 kernel, sm89.cuh).
// PV16 = true:  V^T tiles are fp16 (128 bytes per channel row, 16-byte chunks swizzled by slot = chunk ^ ((d >> 1) & 7)), P is
//               rounded to fp16 and the denominator sums the ROUNDED P in binary32 (what the SageAttention1 kernel's row
//               sum on the tensor cores computes, qk_int_sv_f16_cuda_sm80.cuh:339-368, attn_utils.cuh:599-626).  The PV product is
//               accumulated in fp32; the reference accumulates each 64-key block in fp16 before adding it to its fp32
//               accumulator (attn_utils.cuh:683-751), a rounding this kernel does not reproduce.
// SEL: rows of at most 64 SEL blocks are selected here, by the workgroup that then works on them, instead of by a kernel in
// front that writes a LUT: the row's map is one or two 64-bit scalars, and the next block is its next set bit.  Takes a launch
// (about 4.5 us) and the selection kernel's 7-15 us out of the chain and puts about 3 us in (SPG_SELECT_IN_ATTN_NK: where the line lies).
// G: groups of four wavefronts that share one Q block.  G = 1 is the general kernel.  G > 1 is for grids that leave a row
// alone on its CU (launch_attn): one wavefront per SIMD then waits out every latency of the chain scores - maximum -
// exponentials - product by itself.  The groups take the blocks of the row in turn (group g: places g, g + G, ... of the
// list), each with its own tile rings; what keeps the arithmetic that of the sequential walk is that P is rounded against the
// running maximum of the blocks BEFORE it in the list, so the groups exchange their block maxima through LDS once per round
// of G blocks (at the barrier that the rings need anyway), and so the PV-skip test sees the same differences.  O and the
// denominator are per group and meet in the epilogue.
// FQ: 0 Q comes as INT8 codes and scales; 1 the workgroup quantises its Q block itself; 2 it pools it, too, and works out its similarity
// flag, for a selection in place (SEL).  Codes, pooled row and flag stay in LDS: what a kernel in front would write (half of Q's bytes
// and more) and this one read again.
// SPLIT: a row's blocks go over several workgroups, each with a stretch of its list (launch_split has the why).
template <int D, int ODT, bool PV16, int SEL, int G, int FQ, bool SPLIT>
__global__ __launch_bounds__(256 * G, G == 1 ? 3 : G) void block_sparse_attn_kernel(const AttnParams p) {
  constexpr int KS = D / 32;        // k-steps of the int8 MFMA
  constexpr int NDT = D / 32;       // 32-channel output tiles
  constexpr int TILE = 64 * D;      // bytes of one K tile
  constexpr int VTILE = PV16 ? 2 * TILE : TILE;   // bytes of one V^T tile
  constexpr int CPR = D / 16;       // 16-byte chunks per K row
  constexpr int WL = D / 64;        // global_load_lds instructions per wave per K tile (TILE / 1024 / 4)
  constexpr int WLV = VTILE / 4096; // ... per V^T tile
  // Tile rings.  FP8 PV: three slots each, the tiles of block it+2 are requested while block it is computed.
  // FP16 PV (tiles twice as large): two slots each, so that three workgroups still share a CU (48 KiB): the K tile of
  // block it+2 goes to the slot block it's K tile just left, the V^T tile of block it+1 to the slot of block it-1.
  // With groups the CU holds one workgroup only, and three slots each fit for both.
  constexpr int NBUF = PV16 && G == 1 ? 2 : 3;
  // LDS: per group K ring [NBUF][TILE] | V^T ring [NBUF][VTILE]; votes
  __shared__ __align__(1024) unsigned char smem[G * NBUF * (TILE + VTILE)];
  // PV-skip vote of the per-block mode: a wavefront that votes "skip" stamps the iteration number into its slot; a slot
  // that does not hold the current iteration number means "compute".  Only "skip" votes are written (they are rare at the
  // thresholds in use), and only a wavefront that voted "skip" itself has to read the others' slots.  Two sets of slots,
  // used alternately: a wavefront can be at most one barrier ahead of the slowest one.
  __shared__ int sSkipAt[2][4];
  __shared__ __align__(16) float sVscale[PV16 ? 4 : D];   // fetched at the start, read in the epilogue
  // Groups: block maxima of a round and the running maximum in front of it, one value per query, two sets used alternately.
  __shared__ float sFm[2][G > 1 ? G + 1 : 1][G > 1 ? 128 : 1];
  const int tid = threadIdx.x, lane = tid & 63, r = lane & 31, hh = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(G == 1 ? tid >> 6 : (tid >> 6) & 3);   // uniform: everything derived from it stays scalar
  const int grp = G == 1 ? 0 : __builtin_amdgcn_readfirstlane(tid >> 8);
  unsigned char *const sKr = smem + grp * (NBUF * (TILE + VTILE));
  unsigned char *const sVr = sKr + NBUF * TILE;
  const uint32_t lds_k0 = (uint32_t)(size_t)(__attribute__((address_space(3))) unsigned char *)smem + (uint32_t)(grp * (NBUF * (TILE + VTILE)));   // LDS byte address
  const uint32_t lds_v0 = lds_k0 + NBUF * TILE;

  // A row that is not in its loop yet leaves the matrix units idle: at the loop's own priority its selection takes half as long beside two
  // other rows (8.8 us, 4.3), at the expense of those.  That pays with a LUT, where the start is short, on any grid, and with a selection in
  // place where a few rows more than there are places start when little else runs.  Where all rows start at once there is nothing to gain (24 x
  // 2351 71.0 / 71.2); on larger grids gains and losses are even, but for those of up to two rounds with a partial last Q block: its rows keep all
  // their blocks, begin first and end last, and every row that starts beside them makes them later.  us per call with the priority from
  // the loop on / from here, top-k at D = 128 unless noted, H x N: CDF with similarity 32 x 4096 224.0 / 215.6, GQA 32/8 x 4096 causal 100.5 / 99.7,
  // 16 x 8190 x 2500 102.7 / 101.9, 24 x 4480 125.3 / 117.5, 24 x 4401 129.6 / 125.8, 48 x 2560 99.3 / 95.3; 32 x 4608 147.3 / 146.0, 24 x 7424 232.2 / 232.3, 24 x
  // 5553 166.1 / 170.6, 24 x 7345 254.7 / 263.6, 32 x 5553 203.3 / 217.5, 48 x 3633 158.2 / 167.6, FP16 PV 24 x 5414 239.6 / 250.3; LUT 30 x 17776 D64 1010 /
  // 1008, 16 x 11000 D64 195.9 / 189.9, D128 294.7 / 292.6.
  if constexpr (G == 1)
    if (SEL == 0 || (p.total_wg > 8 * SPG_PLACES && p.total_wg <= SPG_START_PRIO_MAX)) __builtin_amdgcn_s_setprio(3);
  int bh, qb, item = blockIdx.x;
  static_assert(!SPLIT || (SEL == 0 && G == 1 && FQ == 0), "rows in chunks come with a list and with codes of Q");
  int chunk = 0;
  int chunks = 1, chunk_begin = 0, chunk_end = 0;
  if constexpr (SPLIT) {
    if (!place_part(p, item, bh, qb, chunk)) return;
  } else if constexpr (SEL == 0) {                    // (short rows: the grid is over before the XCDs drift apart)
    if (p.queue != nullptr) {
      __shared__ int sItem;
      if (threadIdx.x == 0) sItem = take_item(p, item);
      __syncthreads();
      item = __builtin_amdgcn_readfirstlane(sItem);
      if (item < 0) return;
    }
  }
  if constexpr (!SPLIT)
    if (!place_workgroup(p, item & 7, item >> 3, bh, qb)) return;
  const int batch = p.by_H(bh), head = bh - batch * p.H;
  // grouped-query attention: H / Hkv consecutive query heads share one K/V head (sm89.cuh:118, head_id / num_kv_groups)
  const int bhk = batch * p.Hkv + p.by_group(head);

  const int N = p.N, Nk = p.Nk;
  if constexpr (!PV16 && FQ == 0) fp8_saturation_on();

  // Everything whose address follows from the launch arguments is requested before the first wait: the count, the first
  // four LUT entries (indices clamped to the row, unused ones ignored), the scales, Q.  A chain of dependent scalar loads
  // costs a short row more than its first block.
  // LUT and K scales are read through the constant address space: uniform addresses become scalar loads (SMEM),
  // which never touch the vector-memory counter the tile ring is synchronised with.
  typedef const __attribute__((address_space(4))) int32_t *c_i32_t;
  typedef const __attribute__((address_space(4))) float *c_f32_t;
  const size_t row_id = (size_t)bh * p.nq + qb;
  const int32_t *list = p.lut + (SEL > 0 ? 0 : row_id * p.nk);
  int last_col = p.nk - 1, chunk_first = 0;
  if constexpr (SPLIT) {
    const RowChunks c(((c_i32_t)p.valid)[row_id], p.split);
    if (chunk >= (int)c.n) return;
    chunk = c.turned(chunk, qb);
    chunks = (int)c.n;
    chunk_begin = c.begin(chunk);
    chunk_end = c.begin(chunk + 1);
    chunk_first = chunk > 0 ? ((c_i32_t)p.split.first)[row_id * p.split.chunks + chunk] : ((c_i32_t)list)[0];
    list += chunk_begin;
    last_col -= chunk_begin;
  }
  const c_i32_t lutc = (c_i32_t)list;
  int nv, l0, l1, l2, l3;
  if constexpr (SEL == 0 && G > 1) nv = ((c_i32_t)p.valid)[row_id];
  if constexpr (SEL == 0 && G == 1) {
    nv = SPLIT ? chunk_end - chunk_begin : ((c_i32_t)p.valid)[row_id];
    l0 = SPLIT ? chunk_first : lutc[0]; l1 = lutc[min(1, last_col)]; l2 = lutc[min(2, last_col)]; l3 = lutc[min(3, last_col)];
  }
  // per-warp granularity: the 32 query rows of a wavefront are one quantisation group, so the scale stays a scalar
  float qs;
  if constexpr (FQ == 0) qs = ((c_f32_t)p.q_scale)[p.q_per_warp ? row_id * 4 + wave : row_id];
  const float thr = p.pvthr.p != nullptr ? ((c_f32_t)p.pvthr.p)[head] : p.pvthr.v;

  // ---- Q fragment: B operand of S^T = K.Q^T, resident for the whole loop -------------------------------
  v4i qreg[KS];
  if constexpr (FQ == 0) {
    const int q_row = qb * 128 + wave * 32 + r;
#pragma unroll
    for (int ks = 0; ks < KS; ks++) {
      qreg[ks] = (v4i){0, 0, 0, 0};
      if (q_row < N) qreg[ks] = *(const v4i *)(p.q8 + ((size_t)bh * N + q_row) * D + 32 * ks + 16 * hh);
    }
  }
  // Q from the caller's tensor: codes through the ring slot that the first tiles leave free, 64 rows in its K and 64 in its V^T tile (FP16
  // PV: all in a V^T tile)
  static_assert(FQ == 0 || (G == 1 && D == 128), "where it pays (q_in_front)");
  __shared__ float sQscale[FQ > 0 ? 4 : 1];
  __shared__ __align__(16) uint16_t sPoolQ[FQ == 2 ? D : 8];
  __shared__ uint32_t sSimQ;
  auto quantise_q = [&]() __attribute__((always_inline)) {
    if constexpr (FQ > 0) {
      unsigned char *const lo = NBUF == 3 ? sKr + 2 * TILE : sVr + VTILE, *const hi = NBUF == 3 ? sVr + 2 * VTILE : sVr + VTILE + TILE;
      const PsqToLds<D> to = {sPoolQ, &sSimQ, sQscale, lo, hi, p.q_per_warp == 0};
      float simthr = 0.f;
      if constexpr (FQ == 2) simthr = p.q.simthr.at(head);
      psq_core<128, D, ODT, MEAN_NONE, FQ == 2, 32, 256, 128>(p.q.x + (size_t)batch * p.q.st.sb + (size_t)head * p.q.st.sh, p.q.st.sn, nullptr, nullptr, 0,
                                                              simthr, N, qb, bh, sKr, to);
      __syncthreads();
      const unsigned char *const half = (wave < 2 ? lo : hi) + ((wave & 1) * 32 + r) * D;
#pragma unroll
      for (int ks = 0; ks < KS; ks++) qreg[ks] = *(const v4i *)(half + (((2 * ks + hh) ^ PsqToLds<D>::swz(r)) * 16));
      qs = __builtin_bit_cast(float, __builtin_amdgcn_readfirstlane(__builtin_bit_cast(int, sQscale[wave])));
    }
  };
  if constexpr (FQ == 2) quantise_q();
  constexpr int W = SEL > 0 ? SEL : 1;
  uint64_t map[W] = {};                    // SEL: blocks not fetched yet
  if constexpr (SEL > 0) {
    __shared__ uint16_t sScore[64 * W];
    const uint8_t *simk = p.sel.sim_k + (size_t)bhk * p.nk;
    bool row_forced;
    const uint16_t *pool_q;
    if constexpr (FQ == 2) { row_forced = sSimQ == 0; pool_q = sPoolQ; }
    else { row_forced = p.sel.sim_q[row_id] == 0; pool_q = p.sel.pool_q + row_id * D; }
    bool k_dead[W];
#pragma unroll
    for (int t = 0; t < W; t++) k_dead[t] = simk[min(64 * t + lane, last_col)] == 0;
    // 64 columns a turn, the groups take turns
#pragma unroll
    for (int t = 0; t < W; t++) {
      if (G == 1 || t % G == grp) {
        const int col = 64 * t + ((tid & 255) >> 2);
        const uint16_t s16 = pooled_score_4lanes<D, ODT>(pool_q, p.sel.pool_k + ((size_t)bhk * p.nk + min(col, last_col)) * D, tid & 3);
        if ((tid & 3) == 0) sScore[col] = s16;
      }
    }
    __syncthreads();
    const int causal_lim = p.sel.is_causal ? min(p.nk, 2 * (qb + 1)) : p.nk;
    // One wavefront selects for all of them: the others would take its issue slots, and those of the rows beside this one (H2 N1024 D64 17.8
    // us per call / 17.45, H2 N4096 D128 42.5 / 42.0).
    __shared__ uint64_t sMap[W];
    if (wave == 0 && grp == 0) {
      float sc[W];
#pragma unroll
      for (int t = 0; t < W; t++) sc[t] = (64 * t + lane >= causal_lim || k_dead[t]) ? -INFINITY : elem_to_f32<ODT>(sScore[64 * t + lane]);
      select_row<ODT, W>(map, sc, k_dead, p.sel.by_topk, p.sel.level.at(head), p.nk, causal_lim, row_forced, p.sel.sink, lane);
#pragma unroll
      for (int t = 0; t < W; t++)
        if (lane == 0) sMap[t] = map[t];
    }
    __syncthreads();
#pragma unroll
    for (int t = 0; t < W; t++) {
      const uint64_t w = sMap[t];
      map[t] = (uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)(w >> 32)) << 32 | (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)w);
    }
    nv = 0;
#pragma unroll
    for (int t = 0; t < W; t++) nv += __builtin_popcountll(map[t]);
    if (p.sel.valid_out != nullptr && tid == 0) p.sel.valid_out[row_id] = nv;
  }
  auto drop_lowest = [&]() __attribute__((always_inline)) {
    bool below = true;                     // no lower word holds a block
#pragma unroll
    for (int t = 0; t < W; t++) {
      const uint64_t w = map[t];
      map[t] = below ? w & (w - 1) : w;    // (0 stays 0)
      below = below && w == 0;
    }
  };
  // SEL: takes the next block (of this group) out of the map; beyond the last one it repeats `prev`
  auto next_block = [&](int prev) __attribute__((always_inline)) {
    int b = prev;
#pragma unroll
    for (int t = W - 1; t >= 0; t--) b = map[t] != 0 ? 64 * t + __builtin_ctzll(map[t]) : b;
#pragma unroll
    for (int i = 0; i < G; i++) drop_lowest();
    return b;
  };
  if constexpr (SEL > 0 && G > 1)
    for (int i = 0; i < grp; i++) drop_lowest();
  if (nv == 0) return;                                       // output rows stay unwritten (sm89.cuh:232-235)

  const int8_t *kbase = p.k8 + (size_t)bhk * Nk * D;
  const uint8_t *vbase = p.v8 + (size_t)bhk * p.nk * (size_t)VTILE;
  const c_f32_t kscale = (c_f32_t)(p.k_scale + (size_t)bhk * p.nk);
  const float c = p.sm_scale_log2;

  // ---- tile loader: wave w copies LDS bytes [1024*(WL*w+u), +1024) of each tile, lane l the 16-byte chunk l ----
  // K: LDS chunk position pos <-> (row = pos / CPR, slot = pos % CPR) holds global chunk slot ^ k_swz(row).
  // A tile's global address is (uniform base of the block) + (per-lane 32-bit offset) + u*1024, and the same
  // u*1024 is the LDS offset: it rides in the instruction's immediate (applied to both addresses).
  // The base is a 64-bit shift of the block number: the tiles of one head may span more than 4 GiB.
  // (the two per-lane offsets are recomputed from the thread id where they are used: cheaper than keeping them
  //  in registers across the loop, where the register file is the scarce resource)
  // Split into a part that depends on the lane only (recomputed with three or four vector instructions where it is
  // used) and a wavefront-uniform part that the compiler keeps in scalar registers: the K-row swizzle of chunk position
  // pos = WL*64*wave + lane takes its bits from lane bits 4-5 (D = 128) or 4 (D = 64) and from bit 1 of the wave index.
  static_assert(D == 64 || D == 128, "swizzle bit positions below");
  const uint32_t kswz_wave16 = (uint32_t)((wave >> 1) & 1) << (D == 128 ? 6 : 5);
  const uint32_t k_wave = (uint32_t)(WL * 1024 * wave), v_wave = (uint32_t)(WLV * 1024 * wave);
#define SPG_LANE_OFFSETS()                                                                                    \
  uint32_t lane_ = threadIdx.x & 63u;                                                                         \
  asm volatile("" : "+v"(lane_));                                                                             \
  const uint32_t pos0 = (uint32_t)(WL * 64 * wave) + lane_;                                                   \
  const uint32_t v_lane = v_wave + lane_ * 16u;                                                               \
  const uint32_t kswz_lane = D == 128 ? ((lane_ >> 4) & 3u) : ((lane_ >> 4) & 1u);                            \
  const uint32_t k_lane = k_wave + (((lane_ ^ kswz_lane) << 4) ^ kswz_wave16);   /* row * D + (slot ^ swz) * 16 */
  // FP8 PV, D = 128 or groups: a wavefront copies half of ONE of the two tiles instead of a quarter of each - wavefronts 0 and 1
  // the K tile, 2 and 3 the V^T tile: one base address, one LDS base and one resident lane offset for all its loads of a block.
  // us per call, quarters / halves: H32 N32768 D128 causal 3926 / 3895, one head N17776 D64 (three groups) 170.2 / 168.9; but a mask
  // over H48 N16384 D64 904 / 918, where a wavefront has two loads per block only.
  constexpr bool HALF_LOADS = !PV16 && (D == 128 || G > 1);
  constexpr int HALF = TILE / 2;
  const uint32_t half_swz = wave >= 2 ? 0u : D == 128 ? ((lane >> 4) & 3u) | ((uint32_t)wave << 2) : ((lane >> 4) & 1u) | ((uint32_t)wave << 1);
  const uint32_t half_lane = ((uint32_t)lane ^ half_swz) << 4;
  const uint8_t *const half_base = (wave >= 2 ? vbase : (const uint8_t *)kbase) + (wave & 1) * HALF;
  unsigned char *const half_lds = (wave >= 2 ? sVr : sKr) + (wave & 1) * HALF;
  const int last_partial_blk = (Nk % 64) && (!HALF_LOADS || wave < 2) ? p.nk - 1 : -1;   // the only block with rows beyond Nk
  typedef __attribute__((address_space(3))) void *lds_ptr_t;
  typedef const __attribute__((address_space(1))) void *glb_ptr_t;
#define SPG_LOAD_K_(BLK, KOFF, CHK)   /* inside a scope that holds SPG_LANE_OFFSETS() */                            \
  {                                                                                                           \
    const int8_t *kb_ = kbase + (size_t)(uint32_t)(BLK) * TILE;                                                 \
    unsigned char *lk_ = sKr + (KOFF) + WL * wave * 1024;                                                     \
    if (CHK == 0 || (BLK) != last_partial_blk) {                                                              \
      /* the loads of one tile back to back: they share the LDS base register (M0) */                          \
      __builtin_amdgcn_global_load_lds((glb_ptr_t)(kb_ + k_lane), (lds_ptr_t)lk_, 16, 0, 0);                  \
      if constexpr (WL == 2)                                                                                  \
        __builtin_amdgcn_global_load_lds((glb_ptr_t)(kb_ + k_lane), (lds_ptr_t)lk_, 16, 1024, 0);             \
    } else {                                                                                                  \
      /* rows beyond Nk are clamped to row Nk-1: their scores are masked, their V rows are zero */              \
      const int rows_ok_ = Nk - (BLK) * 64;                                                                    \
      _Pragma("unroll") for (int u = 0; u < WL; u++) {                                                        \
        const uint32_t pos = pos0 + u * 64;                                                                   \
        const uint32_t row_ = min(pos / CPR, (uint32_t)(rows_ok_ - 1));                                       \
        const uint32_t ko_ = row_ * D + (((pos % CPR) ^ k_swz<D>(pos / CPR)) * 16u);                          \
        __builtin_amdgcn_global_load_lds((glb_ptr_t)(kb_ + ko_), (lds_ptr_t)(lk_ + u * 1024), 16, 0, 0);      \
      }                                                                                                       \
    }                                                                                                         \
  }
#define SPG_LOAD_V_(BLK, VOFF)                                                                                \
  {                                                                                                           \
    const uint8_t *vb_ = vbase + (size_t)(uint32_t)(BLK) * VTILE;                                               \
    unsigned char *lv_ = sVr + (VOFF) + WLV * wave * 1024;                                                    \
    __builtin_amdgcn_global_load_lds((glb_ptr_t)(vb_ + v_lane), (lds_ptr_t)lv_, 16, 0, 0);                    \
    if constexpr (WLV >= 2)                                                                                   \
      __builtin_amdgcn_global_load_lds((glb_ptr_t)(vb_ + v_lane), (lds_ptr_t)lv_, 16, 1024, 0);               \
    if constexpr (WLV == 4) {                                                                                 \
      __builtin_amdgcn_global_load_lds((glb_ptr_t)(vb_ + v_lane), (lds_ptr_t)lv_, 16, 2048, 0);               \
      __builtin_amdgcn_global_load_lds((glb_ptr_t)(vb_ + v_lane), (lds_ptr_t)lv_, 16, 3072, 0);               \
    }                                                                                                         \
  }
#define SPG_LOAD_K(BLK, KOFF) { SPG_LANE_OFFSETS() (void)v_lane; SPG_LOAD_K_(BLK, KOFF, 1) }
#define SPG_LOAD_V(BLK, VOFF) { SPG_LANE_OFFSETS() (void)k_lane; (void)pos0; SPG_LOAD_V_(BLK, VOFF) }
// rings of three slots: both tiles of one block into ring slot offset BUFOFF (in K-tile units)
#define SPG_LOAD_QUARTERS(BLK, BUFOFF, CHK) { SPG_LANE_OFFSETS() SPG_LOAD_K_(BLK, BUFOFF, CHK) SPG_LOAD_V_(BLK, (VTILE / TILE) * (BUFOFF)) }
  auto load_tiles = [&](int b, uint32_t boff, auto chk) __attribute__((always_inline)) {
    if constexpr (!HALF_LOADS) { SPG_LOAD_QUARTERS(b, boff, decltype(chk)::value) }
    else {
      const uint8_t *const tb = half_base + (size_t)(uint32_t)b * TILE;
      unsigned char *const tl = half_lds + boff;
      uint32_t lane_off = half_lane;
      if constexpr (decltype(chk)::value || G > 1) asm volatile("" : "+v"(lane_off));   // keeps address arithmetic out of the registers of the loop
      if (!decltype(chk)::value || b != last_partial_blk) {
        __builtin_amdgcn_global_load_lds((glb_ptr_t)(tb + lane_off), (lds_ptr_t)tl, 16, 0, 0);
        __builtin_amdgcn_global_load_lds((glb_ptr_t)(tb + lane_off), (lds_ptr_t)tl, 16, 1024, 0);
        if constexpr (D == 128) {
          __builtin_amdgcn_global_load_lds((glb_ptr_t)(tb + lane_off), (lds_ptr_t)tl, 16, 2048, 0);
          __builtin_amdgcn_global_load_lds((glb_ptr_t)(tb + lane_off), (lds_ptr_t)tl, 16, 3072, 0);
        }
      } else {
        // K rows beyond Nk are clamped to row Nk-1: their scores are masked, their V rows are zero
        const uint8_t *const kb = (const uint8_t *)kbase + (size_t)(uint32_t)b * TILE;
        const uint32_t last_row = (uint32_t)(Nk - 1 - b * 64);
#pragma unroll
        for (int u = 0; u < HALF / 1024; u++) {
          const uint32_t row = (uint32_t)((wave & 1) * 32 + u * (64 / CPR)) + (lane_off / D);   // the swizzle stays within a row
          const uint32_t off = min(row, last_row) * D + (lane_off & (D - 1));
          __builtin_amdgcn_global_load_lds((glb_ptr_t)(kb + off), (lds_ptr_t)(tl + u * 1024), 16, 0, 0);
        }
      }
    }
  };
#define SPG_LOAD_TILES(BLK, BUFOFF, CHK) load_tiles(BLK, BUFOFF, std::integral_constant<int, CHK>{})

  // MFMA row i of key tile kt carries key 32*((i>>2)&1) + 16*kt + 4*(i>>3) + (i&3); rows krow0 and krow0+16 have
  // the same swizzle, so tile 1's operand sits 16 rows (16*D bytes) after tile 0's.
  const int krow0 = 32 * ((r >> 2) & 1) + 4 * (r >> 3) + (r & 3);
  const int ksw = k_swz<D>(krow0);
  // K operand of k-step ks (tile 0): chunk (2ks+hh) ^ ksw = ((2ks) ^ (ksw & 6)) | ((hh ^ ksw) & 1), i.e. the LDS
  // byte offset is k_rd_base + ((32*ks) ^ k_rd_x): one xor-add per read, two registers.
  const uint32_t k_rd_base = (uint32_t)(krow0 * D + ((hh ^ ksw) & 1) * 16);
  const uint32_t k_rd_x = (uint32_t)((ksw & 6) * 16);
  const int vsw = v_swz(r);                // v_swz(32*dt + r) does not depend on dt
  // V^T operand: key chunks 2hh and 2hh+1 of channel row r (+32*dt); the two swizzled slots differ in bit 4 only
  const uint32_t v_rd_lo = (uint32_t)(r * 64 + (((2 * hh) ^ vsw) * 16));
  // fp16 V^T operand of key step s: chunk (4hh + s) ^ ((r >> 1) & 7) of the 128-byte row r (+32*dt): v_rd16 ^ (16 * s)
  const uint32_t v_rd16 = (uint32_t)(r * 128 + (((4 * hh) ^ ((r >> 1) & 7)) * 16));

  float m = SPG_NEG_BIG;
  if constexpr (SPLIT) {
    // the running maximum in front of the chunk's first block
    const float *cm = p.split.maxima + row_id * p.split.chunks * 128 + wave * 32 + r;
#pragma unroll 4
    for (int i = 0; i < chunk; i++) m = fmaxf(m, cm[i * 128]);
  }
  // d = 1.0 initially (sm89.cuh:172).  Each half-lane sums its own 32 keys, so only one of the two starts at 1.
  float dsum = hh == 0 && grp == 0 && chunk == 0 ? 1.0f : 0.0f;
  float m_own = SPG_NEG_BIG;               // groups: the maximum that this group's O and dsum refer to
  v16f O[NDT];
#pragma unroll
  for (int dt = 0; dt < NDT; dt++)
#pragma unroll
    for (int e = 0; e < 16; e++) O[dt][e] = 0.f;
  int cnt = 0;

  // block ids: blk = block of iteration it, blk1 = it+1, blk2 = it+2 (tiles in flight); d3 = LUT delta of it+3.
  // K scales are fetched one iteration ahead as well.  With groups an iteration is a round: place it * G + grp of the list.
  int blk, blk1, blk2, d3 = 0;
  if constexpr (SEL == 0 && G > 1) {
    // the LUT holds differences: running sums of its first entries, unused ones read as 0
    int at = 0, acc = 0;
    auto advance = [&](int upto) __attribute__((always_inline)) {
      int l[G];
#pragma unroll
      for (int i = 0; i < G; i++) l[i] = lutc[min(at + i, last_col)];
#pragma unroll
      for (int i = 0; i < G; i++) acc += at + i < min(nv, upto) ? l[i] : 0;
      at = upto;
    };
    advance(grp + 1); blk = acc;
    advance(grp + 1 + G); blk1 = acc;
    advance(grp + 1 + 2 * G); blk2 = acc;
    acc = 0;
    advance(grp + 1 + 3 * G); d3 = acc;
  } else if constexpr (SEL > 0) {
    blk = next_block(0);
    blk1 = next_block(blk);
    blk2 = next_block(blk1);
  } else {
    blk = l0;
    blk1 = blk + (nv > 1 ? l1 : 0);
    blk2 = blk1 + (nv > 2 ? l2 : 0);
    d3 = nv > 3 ? l3 : 0;
  }
  float ksc = kscale[blk], ksc1 = kscale[blk1];
  if constexpr (PV16 && G == 1) {
    SPG_LOAD_K(blk, 0);
    SPG_LOAD_V(blk, 0);
    if (nv > 1) SPG_LOAD_K(blk1, TILE);           // the V^T tile of block 1 follows behind the first barrier
  } else {
    SPG_LOAD_TILES(blk, 0, 1);
    if (nv > grp + G) SPG_LOAD_TILES(blk1, TILE, 1);
  }
  if constexpr (!PV16) {
    if (wave < D / 64 && grp == 0)
      __builtin_amdgcn_global_load_lds((glb_ptr_t)(p.v_scale + (size_t)bhk * D + wave * 64 + lane), (lds_ptr_t)(sVscale + wave * 64), 4, 0, 0);
  }
  if constexpr (FQ == 1) quantise_q();
  if constexpr (!PV16 && FQ > 0) fp8_saturation_on();   // (behind the conversions of Q, whose overflows stay infinite)
  uint32_t bufoff = 0;                     // LDS ring offset of block it

  // The INT8 accumulators do not start at zero but at the bit pattern 0x3E22F983 - the float 1/(2 pi), which the
  // instruction set offers as an INLINE CONSTANT, so the first product of each chain takes it as its C operand and no
  // register has to be initialised.  Its mantissa field is 2 292 099 and |dot| <= 128 * 128 * 128 = 2 097 152, so
  // the int32 sum stays inside the binade [1/8, 1/4): the accumulator READ AS A FLOAT is exactly
  // 1/(2 pi) + dot * 2^-26, and the scores need no int-to-float conversion - the 2^26 goes into the multiplier and the
  // constant into the additive term of the fma that feeds exp2.
  const float acc_c = __builtin_bit_cast(float, (int)SPG_ACC_C_BITS);
  if (tid < 8) (&sSkipAt[0][0])[tid] = -1;   // no slot may hold an iteration number by accident
  __builtin_amdgcn_s_waitcnt(0x0F70);     // vmcnt(0): Q fragment and the first tiles have arrived
  __syncthreads();

  // One K block.  TAIL = false: every block but the last two - PV-threshold test, no masks (sm89.cuh:283-391).
  // TAIL = true: the last two blocks - token-causal and out-of-bound masks where a score needs them, no skip
  // (sm89.cuh:467-648).  The two are
  // separate loops so that the common one carries none of the tail's predicates.
  // SLOT = 0, 1, 2: the ring slot of the block is a compile-time constant (the common loop is unrolled over the ring), so
  // every LDS address of the iteration is a loop-invariant register plus an immediate offset; SLOT = -1: the slot is the
  // run-time value `bufoff` (the left-over blocks of the common loop and the two tail blocks).
  uint32_t kaddr_c[KS];
#pragma unroll
  for (int ks = 0; ks < KS; ks++) kaddr_c[ks] = lds_k0 + k_rd_base + ((uint32_t)(32 * ks) ^ k_rd_x);
  const uint32_t va_lo_c = lds_v0 + v_rd_lo, va_hi_c = lds_v0 + (v_rd_lo ^ 16u);
  const float cq26 = c * qs * SPG_ACC_SCALE;        // exponent multiplier a of a block = cq26 * k_scale * 2^-26
  // a 2^26 / (2 pi) >= 2^14  <=>  k_scale >= this bound; both are positive floats, so their bit patterns compare as integers
  const int kscale_precise_bits = __builtin_bit_cast(int, 16384.0f / (acc_c * cq26));
  auto step = [&](auto tail_tag, auto slot_tag, const int it) __attribute__((always_inline)) {
    constexpr bool TAIL = decltype(tail_tag)::value;
    constexpr int SLOT = decltype(slot_tag)::value;
    constexpr bool CS = SLOT >= 0;                  // compile-time ring slot
    const int place = G == 1 ? it : it * G + grp;   // in the row's list of blocks
    // groups: a round at the end can hold ordinary blocks, the last two and places beyond the list side by side
    const bool tail = TAIL && (G == 1 || place >= nv - 2), active = !TAIL || G == 1 || place < nv;
    // ---- S^T = K . Q^T ---------------------------------------------------------------------------------
    v16i S0, S1;
    {
      // two groups of k-steps: the reads of the second group are in flight while the first group's MFMAs run
      constexpr int HK = KS / 2;
      v4i a0[KS], a1[KS];
      auto read_k = [&](int ks) __attribute__((always_inline)) {
        if constexpr (CS) lds_read_2x128<(SLOT < 0 ? 0 : SLOT) * TILE, (SLOT < 0 ? 0 : SLOT) * TILE + 16 * D>(a0[ks], a1[ks], kaddr_c[ks]);
        else lds_read_2x128<0, 16 * D>(a0[ks], a1[ks], kaddr_c[ks] + bufoff);
      };
      // FP16 PV: two k-steps in registers, each replaced by the one after next as soon as its products are issued
      if constexpr (PV16) {
        read_k(0); read_k(1);
        lds_wait_but<2>(a0[0], a1[0]);
        asm volatile("v_mfma_i32_32x32x32_i8 %0, %2, %4, 0.15915494\n\tv_mfma_i32_32x32x32_i8 %1, %3, %4, 0.15915494"
                     : "=&v"(S0), "=&v"(S1)
                     : "v"(a0[0]), "v"(a1[0]), "v"(qreg[0]));
#pragma unroll
        for (int ks = 1; ks < KS; ks++) {
          __builtin_amdgcn_sched_barrier(0);
          if (ks + 1 < KS) { read_k(ks + 1); lds_wait_but<2>(a0[ks], a1[ks]); }
          else lds_wait_but<0>(a0[ks], a1[ks]);
          S0 = __builtin_amdgcn_mfma_i32_32x32x32_i8(a0[ks], qreg[ks], S0, 0, 0, 0);
          S1 = __builtin_amdgcn_mfma_i32_32x32x32_i8(a1[ks], qreg[ks], S1, 0, 0, 0);
        }
      } else {
      // first group: nothing to overlap with, the reads carry their wait
      {
        constexpr int SO = CS ? SLOT * TILE : 0;
        const uint32_t bo = CS ? 0u : bufoff;
        if constexpr (HK == 2) lds_read_4x128_wait<SO, SO + 16 * D>(a0[0], a1[0], a0[1], a1[1], kaddr_c[0] + bo, kaddr_c[1] + bo);
        else lds_read_2x128_wait<SO, SO + 16 * D>(a0[0], a1[0], kaddr_c[0] + bo, kaddr_c[0] + bo);
      }
      // second group: in flight under the first group's products
#pragma unroll
      for (int ks = HK; ks < KS; ks++) read_k(ks);
      // the first product of each chain, with the inline constant as its C operand (the compiler would otherwise keep
      // the constant in sixteen registers); the products that follow accumulate onto these and are ordinary builtins,
      // which the other chain's product always separates from their predecessor
      asm volatile("v_mfma_i32_32x32x32_i8 %0, %2, %4, 0.15915494\n\tv_mfma_i32_32x32x32_i8 %1, %3, %4, 0.15915494"
                   : "=&v"(S0), "=&v"(S1)
                   : "v"(a0[0]), "v"(a1[0]), "v"(qreg[0]));
#pragma unroll
      for (int ks = 1; ks < HK; ks++) {
        S0 = __builtin_amdgcn_mfma_i32_32x32x32_i8(a0[ks], qreg[ks], S0, 0, 0, 0);
        S1 = __builtin_amdgcn_mfma_i32_32x32x32_i8(a1[ks], qreg[ks], S1, 0, 0, 0);
      }
      if constexpr (HK == 2) lds_wait4(a0[2], a1[2], a0[3], a1[3]); else lds_wait2(a0[1], a1[1]);
#pragma unroll
      for (int ks = HK; ks < KS; ks++) {
        S0 = __builtin_amdgcn_mfma_i32_32x32x32_i8(a0[ks], qreg[ks], S0, 0, 0, 0);
        S1 = __builtin_amdgcn_mfma_i32_32x32x32_i8(a1[ks], qreg[ks], S1, 0, 0, 0);
      }
      }
    }

    // scalar prefetches for later iterations (SMEM).  Issued here, behind the last LDS wait of the products: scalar and
    // LDS loads share one counter, so a scalar load issued at the top of the loop would be waited for together with the
    // K operands; from here its latency runs under the MFMAs and the max reduction.
    __builtin_amdgcn_sched_barrier(0);
    float ksc2 = 0.f;
    int d4 = 0, d4g[G] = {};
    if constexpr (!TAIL || G > 1) {
      ksc2 = *(c_f32_t)((const __attribute__((address_space(4))) char *)kscale + (uint32_t)(blk2 << 2));
      if constexpr (SEL == 0 && G == 1) d4 = it + 4 < nv ? lutc[(uint32_t)(it + 4)] : 0;
      if constexpr (SEL == 0 && G > 1) {
#pragma unroll
        for (int i = 0; i < G; i++) d4g[i] = place + 3 * G + 1 + i < nv ? lutc[(uint32_t)(place + 3 * G + 1 + i)] : 0;
      }
    }
    __builtin_amdgcn_sched_barrier(0);
    const float dq = qs * ksc;                     // used by the tail blocks only
    // S0/S1 are never rewritten (no copies at the join of the two paths): slot e < 16 is S0[e], slot e >= 16 is S1[e - 16]
    // multiplier of the accumulator read as a float: a * 2^26.  Wavefront-uniform, but kept in a vector register: with two or
    // more wavefronts per SIMD a multiply-add of three vector registers issues in 2.6 clocks, one that reads a scalar register
    // in 4.3 (128 of them per wavefront, three wavefronts: 138 against 233 ns)
    const float a26 = cq26 * ksc;
    // The constant 1/(2 pi) leaves the exponent through ONE additive term, -(1/(2 pi) a 2^26 + m) (+ 8.807), whose rounding
    // error is half an ulp of 1.07e7 a.  Below 2^14 that is at most 2^-11 in the exponent (3e-4 relative in P, and the
    // row maximum's P stays below 448.2).  At or above it (large |q| |k| or a large softmax scale; uniform for the
    // wavefront) the scores are first taken relative to the lane's own maximum - an exact subtraction inside one binade -
    // so that no large constant is left to round: one more instruction per score, on such blocks only.
    const bool precise = __builtin_bit_cast(int, ksc) >= kscale_precise_bits;
    float fm, mloc = acc_c;
    int lim = 0x7fffffff;
    // The last two blocks take the masked arithmetic only if some score of the wavefront is masked at all (token-causal
    // kernels near the diagonal, a partial last K block); otherwise they run the arithmetic of the common loop, which
    // differs from the reference's masked branch (de-quantise, then scale) by the order of two binary32 roundings.
    bool masked = false;                             // wavefront-uniform
    if constexpr (TAIL) {
      // slot e of this lane is key 64*blk + 32*hh + e; keys beyond `lim` are masked
      uint32_t t = threadIdx.x;                                  // (the lane is worked out here: no register holds it across the loop)
      asm volatile("" : "+v"(t));
      const int key0 = blk * 64 + (int)(t & 32u), row = qb * 128 + wave * 32 + (int)(t & 31u);
      if (p.is_causal) lim = row - key0;                         // key > query (attn_utils.cuh:334-361)
      if (place == nv - 1) lim = min(lim, Nk - 1 - key0);        // key >= kv_len (attn_utils.cuh:363-389)
      masked = tail && __any(lim < 31);
    }
    if (!masked) {
      int imax = S0[0];
#pragma unroll
      for (int e = 1; e < 16; e++) imax = max(imax, S0[e]);
#pragma unroll
      for (int e = 0; e < 16; e++) imax = max(imax, S1[e]);
      mloc = __builtin_bit_cast(float, imax);   // 1/(2 pi) + 2^-26 * the largest of this lane's 32 dot products
      fm = (mloc - acc_c) * a26;                // the subtraction is exact (same binade)
    } else {
      fm = SPG_NEG_BIG;
      const float dq26 = dq * SPG_ACC_SCALE;
#pragma unroll
      for (int e = 0; e < 32; e++) {
        float v = (__builtin_bit_cast(float, e < 16 ? S0[e] : S1[e - 16]) - acc_c) * dq26;
        v = e > lim ? SPG_NEG_BIG : v;
        fm = fmaxf(fm, v);
        if (e % 4 == 3) __builtin_amdgcn_sched_barrier(0);   // (one group after the other: the scheduler would spread them over registers that the loop does not have)
      }
      fm = fm * c;
    }
    fm = half_swap_max_raw(fm);
    float diff, m_new, m_old;
    if constexpr (G == 1) {
      diff = fm - m;
      m_new = max_raw(m, fm);
      m_old = m;
      m = m_new;
    } else {
      if (!active) fm = -INFINITY;
      sFm[it & 1][grp][wave * 32 + r] = fm;                      // (both halves hold the same value)
      if (grp == 0) sFm[it & 1][G][wave * 32 + r] = m;
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    }
    int vote = 1;
    if constexpr (!TAIL && G == 1) {
      // max over rows of (diff) + thr > 0  <=>  some row has diff + thr > 0 (fp32 addition is monotonic)
      vote = __any(diff > -thr);          // (the sign of a binary32 sum is exact)
      if (__builtin_expect(vote == 0, 0)) {                    // wavefront-uniform
        sSkipAt[it & 1][wave] = it;       // every lane: a branch on the lane would make the body's control flow divergent
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      }
    }
    __builtin_amdgcn_s_waitcnt(0x0F70);   // this wave's share of block it+1's tiles has landed in LDS
    // block it+1's tiles are complete; the votes are visible; ring slot of block it-1 is free.  (A bare barrier: the fence
    // of __syncthreads() would also wait for the scalar loads above.)
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    bool compute = true;
    if constexpr (G > 1) {
      float before = m, after = -INFINITY;                       // maxima of the round's earlier / later blocks
#pragma unroll
      for (int g = 0; g < G; g++) {
        const float v = sFm[it & 1][g][wave * 32 + r];
        if (g < grp) before = max_raw(before, v);
        if (g > grp) after = max_raw(after, v);
      }
      diff = fm - before;
      m_old = m_own;
      m_new = max_raw(before, fm);
      m = max_raw(m_new, after);
      m_own = m_new;
      if (!TAIL || (active && !tail)) {
        // a wavefront that votes "skip" looks at the other queries of the Q block: their maxima are all here
        if (!__any(diff + thr > 0.f)) {
          bool some = false;
#pragma unroll
          for (int u = 0; u < 2; u++) {
            const int q = lane + 64 * u;
            float b = sFm[it & 1][G][q];
#pragma unroll
            for (int g = 0; g < G - 1; g++) b = g < grp ? fmaxf(b, sFm[it & 1][g][q]) : b;
            some |= sFm[it & 1][grp][q] - b + thr > 0.f;
          }
          compute = __any(some);
        }
      }
      if (TAIL) compute = compute && active;
    }
    if constexpr (!TAIL && G == 1) {   // workgroup-uniform in the per-block mode (sm89.cuh:318-353), wavefront-uniform otherwise
      // per-block mode: a wavefront whose own vote is set knows the OR already; only one that voted "skip" has to read
      // what the others wrote (an LDS round trip that the common case does without)
      if (__builtin_expect(vote == 0, 0)) {
        compute = p.pv_mode == 0;
        if (p.pv_mode == 1) compute = !__builtin_amdgcn_readfirstlane(sSkipAt[it & 1][0] == it && sSkipAt[it & 1][1] == it && sSkipAt[it & 1][2] == it && sSkipAt[it & 1][3] == it);
      }
    }
    if constexpr (PV16 && G == 1) {
      // two-slot rings: every wavefront is past its reads of K slot it % 2 (this block's scores) and of V^T slot
      // (it + 1) % 2 (the previous block's P.V product)
      SPG_LANE_OFFSETS()
      (void)pos0;
      const uint32_t here = CS ? (uint32_t)(SLOT * TILE) : bufoff;
      if ((!TAIL && !(SPLIT && !CS)) || it + 2 < nv) SPG_LOAD_K_(blk2, here, (TAIL || SLOT < 0));
      if ((!TAIL && !(SPLIT && !CS)) || it + 1 < nv) SPG_LOAD_V_(blk1, 2 * (here ^ (uint32_t)TILE));
    } else if ((!TAIL && !(SPLIT && !CS)) || place + 2 * G < nv) {
      if constexpr (CS) {
        SPG_LOAD_TILES(blk2, ((SLOT + 2) % 3) * TILE, 0);
      } else {
        const uint32_t b2 = bufoff == 0 ? 2 * TILE : bufoff - TILE;   // slot (it+2) % 3
        SPG_LOAD_TILES(blk2, b2, 1);
      }
    }
    // the running maximum of some query rose: rescale (exp2(0) = 1 exactly, so the other iterations need neither the
    // exponential nor the products).  Only the lanes of such a query take part - mostly one or two of the 32: the clock under
    // this kernel is set by its power, and idle lanes draw none (H32 N32768 D128 causal 3918 -> 3895 us, a mask over H48
    // N16384 D128 1371 -> 1358)
    if (G == 1 ? diff > 0.f : m_new > m_old) {
      const float osc = __builtin_amdgcn_exp2f(m_old - m_new);
      dsum *= osc;
#pragma unroll
      for (int dt = 0; dt < NDT; dt++)
#pragma unroll
        for (int e = 0; e < 16; e++) O[dt][e] *= osc;
    }
    if (__builtin_expect(compute, 1)) {
      cnt++;
      const float neg0 = PV16 ? -m_new : -m_new + SPG_FP8_OFFSET;
      float ps;
      float x[32];
      if (!masked) {
        // three passes kept apart for the scheduler: a multiply-add feeding the exponential of the same element directly,
        // and the exponential feeding the running sum, would issue as one long chain of dependent instructions
        float neg = __builtin_fmaf(-acc_c, a26, neg0);   // takes the accumulator constant out: one rounding per row
        if (__builtin_expect(precise, 0)) {
          // (S - S_max,lane) a + (S_max,lane a - m + offset): what the reference's fma(S, a, -m + offset) computes
          // (attn_utils.cuh:391-415), with the rounding of m as the only error
          neg = __builtin_fmaf(mloc - acc_c, a26, neg0);
#pragma unroll
          for (int e = 0; e < 16; e++) {
            const int s0 = S0[e], s1 = S1[e];
            S0[e] = __builtin_bit_cast(int, __builtin_bit_cast(float, s0) - mloc);
            S1[e] = __builtin_bit_cast(int, __builtin_bit_cast(float, s1) - mloc);
          }
        }
#pragma unroll
        for (int e = 0; e < 16; e++) {
          const int s0 = S0[e], s1 = S1[e];
          S0[e] = __builtin_bit_cast(int, __builtin_fmaf(__builtin_bit_cast(float, s0), a26, neg));
          S1[e] = __builtin_bit_cast(int, __builtin_fmaf(__builtin_bit_cast(float, s1), a26, neg));
        }
      } else {
        const float masked = __builtin_fmaf(SPG_NEG_BIG, c, neg0);   // what the sentinel score turns into
        const float dq26 = dq * SPG_ACC_SCALE;
        // de-quantised score first, then the softmax scale, as the reference's masked branch does (sm89.cuh:467-648)
#pragma unroll
        for (int e = 0; e < 16; e++) {
          const int s0 = S0[e], s1 = S1[e];
          const float t0 = __builtin_fmaf((__builtin_bit_cast(float, s0) - acc_c) * dq26, c, neg0);
          const float t1 = __builtin_fmaf((__builtin_bit_cast(float, s1) - acc_c) * dq26, c, neg0);
          S0[e] = __builtin_bit_cast(int, e > lim ? masked : t0);
          S1[e] = __builtin_bit_cast(int, e + 16 > lim ? masked : t1);
        }
      }
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int e = 0; e < 32; e++) x[e] = __builtin_amdgcn_exp2f(__builtin_bit_cast(float, e < 16 ? S0[e] : S1[e - 16]));
      __builtin_amdgcn_sched_barrier(0);
      if constexpr (!PV16) {
        // (four chains at D = 64, whose two P.V matrix instructions do not cover one chain of 31 dependent additions)
        constexpr int NC = D == 64 ? 4 : 1;
        float pc[NC];
#pragma unroll
        for (int e = 0; e < NC; e++) pc[e] = x[e];
#pragma unroll
        for (int e = NC; e < 32; e++) pc[e % NC] += x[e];
        ps = pc[0];
        if constexpr (NC == 4) ps = (pc[0] + pc[1]) + (pc[2] + pc[3]);
      }
      if constexpr (PV16) {
        typedef _Float16 h8 __attribute__((ext_vector_type(8)));
        typedef _Float16 h2 __attribute__((ext_vector_type(2)));
        typedef float f2 __attribute__((ext_vector_type(2)));
        h8 pb16[4];
#pragma unroll
        for (int s4 = 0; s4 < 4; s4++)
#pragma unroll
          for (int j = 0; j < 8; j += 2) {
            const f2 pr = {x[8 * s4 + j], x[8 * s4 + j + 1]};
            const h2 ph = __builtin_convertvector(pr, h2);          // v_cvt_pk_f16_f32, round to nearest even
            pb16[s4][j] = ph[0];
            pb16[s4][j + 1] = ph[1];
          }
        {
          // row sums of the ROUNDED P (the reference sums them on the tensor cores, rowsum_f16f16f32, attn_utils.cuh:614):
          // v_dot2_f32_f16 with a pair of ones adds two fp16 values to a binary32 accumulator per instruction, which
          // leaves the matrix unit to the two products.  Each half-lane sums its own 32 keys; the halves meet in the
          // epilogue.
          const h2 ones2 = {(_Float16)1, (_Float16)1};
          float rs = 0.f;
#pragma unroll
          for (int s4 = 0; s4 < 4; s4++)
#pragma unroll
            for (int j = 0; j < 8; j += 2) {
              const h2 pr = {pb16[s4][j], pb16[s4][j + 1]};
              rs = __builtin_amdgcn_fdot2(pr, ones2, rs, false);
            }
          dsum += rs;
        }
        // V^T operands: two 16-key steps in registers, each replaced by the one after next as soon as its products are issued.
        // (Two halves of two steps, every read waited for at once: H24 N8192 D128 causal 334 us, so 332; 4 heads N8192, two groups, 98.9 / 97.7.)
        constexpr int SB = CS ? SLOT * VTILE : 0;    // ring slot as an immediate, or in the address register
        const uint32_t va = lds_v0 + v_rd16 + (CS ? 0u : 2 * bufoff);
        v4i t[4][NDT];
        auto read_v = [&](int st) __attribute__((always_inline)) {
          const uint32_t a_ = va ^ (uint32_t)(16 * st);
          if constexpr (NDT == 4) lds_read_4x128<SB, SB + 4096, SB + 8192, SB + 12288>(t[st][0], t[st][1], t[st][2], t[st][3], a_);
          else lds_read_2x128<SB, SB + 4096>(t[st][0], t[st][1], a_);
        };
        auto wait_v = [&](int st, auto but) __attribute__((always_inline)) {
          if constexpr (NDT == 4) lds_wait_but<decltype(but)::value>(t[st][0], t[st][1], t[st][2], t[st][3]);
          else lds_wait_but<decltype(but)::value>(t[st][0], t[st][1]);
        };
        read_v(0); read_v(1);
#pragma unroll
        for (int st = 0; st < 4; st++) {
          if (st < 3) wait_v(st, std::integral_constant<int, NDT>{}); else wait_v(st, std::integral_constant<int, 0>{});
#pragma unroll
          for (int dt = 0; dt < NDT; dt++)
            O[dt] = __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(h8, t[st][dt]), pb16[st], O[dt], 0, 0, 0);
          __builtin_amdgcn_sched_barrier(0);
          if (st < 2) read_v(st + 2);
        }
      } else {
      dsum += ps;
      v8i pb;
#pragma unroll
      for (int u = 0; u < 8; u++) pb[u] = pack4_e4m3(x[4 * u], x[4 * u + 1], x[4 * u + 2], x[4 * u + 3]);
      {
        constexpr int HD = NDT / 2;
        constexpr int SB = CS ? SLOT * TILE : 0;     // ring slot as an immediate, or in the address registers
        const uint32_t va_lo = CS ? va_lo_c : va_lo_c + bufoff, va_hi = CS ? va_hi_c : va_hi_c + bufoff;
        v4i lo[NDT], hi[NDT];
        // group 0 (output tile dt reads channel rows 32 dt .. 32 dt + 31: 2048 bytes further on)
        if constexpr (HD == 2) lds_read_4x128_wait<SB, SB + 2048>(lo[0], lo[1], hi[0], hi[1], va_lo, va_hi);
        else lds_read_2x128_wait<SB, SB>(lo[0], hi[0], va_lo, va_hi);
        // group 1 in flight while group 0 multiplies
        if constexpr (HD == 2) {
          lds_read_pair<SB + 4096>(lo[2], hi[2], va_lo, va_hi);
          lds_read_pair<SB + 6144>(lo[3], hi[3], va_lo, va_hi);
        } else {
          lds_read_pair<SB + 2048>(lo[1], hi[1], va_lo, va_hi);
        }
#pragma unroll
        for (int dt = 0; dt < HD; dt++) {
          const v8i av = {lo[dt][0], lo[dt][1], lo[dt][2], lo[dt][3], hi[dt][0], hi[dt][1], hi[dt][2], hi[dt][3]};
          O[dt] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(av, pb, O[dt], 0, 0, 0, 0, 0, 0);
        }
        if constexpr (HD == 2) lds_wait4(lo[2], hi[2], lo[3], hi[3]); else lds_wait2(lo[1], hi[1]);
#pragma unroll
        for (int dt = HD; dt < NDT; dt++) {
          const v8i av = {lo[dt][0], lo[dt][1], lo[dt][2], lo[dt][3], hi[dt][0], hi[dt][1], hi[dt][2], hi[dt][3]};
          O[dt] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(av, pb, O[dt], 0, 0, 0, 0, 0, 0);
        }
      }
      }   // !PV16
    }
    // the scalar prefetches are taken over here, where no LDS read is in flight: a first use behind the next K reads
    // would wait for those as well (one counter)
    if constexpr (G > 1) {
      asm volatile("" : "+s"(ksc2));
#pragma unroll
      for (int i = 0; i < G; i++) d4 += d4g[i];
    } else if constexpr (!TAIL) {
      if constexpr (SEL > 0) asm volatile("" : "+s"(ksc2));
      else asm volatile("" : "+s"(ksc2), "+s"(d4));
    }
    // advance the block pipeline and the ring
    blk = blk1; blk1 = blk2;
    if constexpr (SEL > 0) blk2 = next_block(blk2);
    else { blk2 = blk2 + d3; d3 = d4; }
    ksc = ksc1; ksc1 = ksc2;
    if constexpr (!CS) bufoff = bufoff == (NBUF - 1) * TILE ? 0 : bufoff + TILE;
  };
  {
    int it = 0;
    // rounds whose successor's successor ends in front of the last block (no partial tile to load); rounds in front of the
    // last two blocks; all rounds
    const int n_fast = G == 1 ? nv - 3 : (nv - 1) / G - 2, n_all = (nv + G - 1) / G;
    const int n_common = G > 1 ? (nv - 2) / G : SPLIT && chunk < chunks - 1 ? nv : nv - 2;   // (only a row's last two blocks are masked)
    // the common loop, one block per ring slot and trip; the slots are compile-time constants and `bufoff` stays 0.  (FP16 PV with
    // run-time slots: H24 N8192 D128 causal 333 us, so 329; H6 N16384 381 / 377, H10 N5000 122 / 120, H1 N12000 D64 121 / 119.)
    // The wavefronts of a SIMD are served oldest first: of the three rows on a CU the first runs at almost the speed it would
    // have alone, the last gets what is left and ends alone, at less than half the rate of three (three rows of 32 blocks ended
    // at 50, 67 and 83 us).  While other rows wait for a place that is welcome.  The rows of an XCD that none wait for lower
    // their priority as they near their end, so that those with more to do catch up and all end together.  us per call
    // without / with, H x N top-k 0.5: D128 6 x 8192 124 / 118, 13 x 8192 214 / 201, 20 x 8192 272 / 263, 26 x 8192 354 / 342, causal 28 x
    // 4096 118 / 116, D64 14 x 8192 156 / 144, 30 x 17776 1035 / 1016, FP16 PV 6 x 16384 379 / 367.  (The last 64 or 80 rows
    // instead of the places of an XCD: 13 x 8192 205 / 200, 20 x 8192 266 / 267; steps at thirds of the row: 205, 265.)
    // The priority counts against every wavefront of the SIMD, those of other streams' kernels among them, as long as a row runs.  Raised for
    // the last 192 rows of an XCD only, which alone meet the ones that lower theirs, calls are slower (30 x 17776 D64 top-k 1026 / 1048, CDF
    // 1851 / 1915), and what else runs gains nothing by it: three wavefronts of 168 registers leave no room on a SIMD, and beside D64 48 x 16384
    // small kernels of another stream take as long either way (an addition over a million floats 54.6, 51.5 with priority and 50.5, 51.4
    // without, 4.5 us alone).
    // Rows in chunks: `item` counts chunks, wg_per_xcd rows, so up to 768 rows every chunk lowers its priority, also one that others wait for:
    // the chunks of a round end together and the next ones start together.  Beyond 768 rows the first of an XCD do not.  us per call so /
    // without lower priorities / over the last 96 chunks of an XCD only, top-k:
    //   D64   H1 N17776 0.5 90.0 / 92.7 / 92.6, H4 N17776 0.15 127.1 / 135.9 / 135.6, H1 N30001 0.3 136.4 / 147.3 / 147.3
    //   D128  H1 N17776 0.5 124.8 / 129.5 / 129.1, H2 N17776 0.5 205.6 / 202.6 / 202.0, H1 N30001 0.3 193.1 / 209.9 / 206.6
    //   FP16 PV, D128  H2 N17776 0.5 238.5 / 232.5 / 232.7
    // and so / all of them, H8 N17776 0.15, 1112 rows: D64 185.8 / 202.7, D128 279.5 / 269.8.
    int drop_at = 0x7fffffff;
    if constexpr (G == 1) {
      __builtin_amdgcn_s_setprio(3);
      if ((item >> 3) >= p.wg_per_xcd - SPG_PLACES) drop_at = nv >> 1;
    }
#pragma unroll 1
    for (; it + NBUF <= n_fast; it += NBUF) {
      if constexpr (G == 1) {
        if (it >= drop_at) {
          const int d2 = nv - (nv >> 2), d3 = nv - (nv >> 3);
          __builtin_amdgcn_s_setprio(2);
          if (it >= d2) __builtin_amdgcn_s_setprio(1);
          if (it >= d3) __builtin_amdgcn_s_setprio(0);
          drop_at = it >= d3 ? 0x7fffffff : it >= d2 ? d3 : d2;
        }
      }
      step(std::false_type{}, std::integral_constant<int, 0>{}, it);
      step(std::false_type{}, std::integral_constant<int, 1>{}, it + 1);
      if constexpr (NBUF == 3) step(std::false_type{}, std::integral_constant<int, 2>{}, it + 2);
    }
#pragma unroll 1
    for (; it < n_common; it++) step(std::false_type{}, std::integral_constant<int, -1>{}, it);
#pragma unroll 1
    for (; it < n_all; it++) step(std::true_type{}, std::integral_constant<int, -1>{}, it);
  }
#undef SPG_LOAD_TILES
#undef SPG_LOAD_QUARTERS
#undef SPG_LOAD_K
#undef SPG_LOAD_V
#undef SPG_LOAD_K_
#undef SPG_LOAD_V_
#undef SPG_LANE_OFFSETS

  // one count per wavefront of 32 query rows, the layout of the reference's PV_Count (sm89.cuh:650-659); the four
  // counts of a Q block are equal because the skip decision is taken per block
  if (p.pv_count != nullptr && lane == 0) p.pv_count[((size_t)bh * p.nq + qb) * 4 + wave] = cnt;

  // ---- epilogue: O / d * v_scale -> out dtype -----------------------------------------------------------
  if constexpr (SPLIT) {
    // (worked out again: no register holds them across the loop)
    int id = blockIdx.x;
    asm volatile("" : "+s"(id));
    const size_t row_id = (size_t)bh * p.nq + qb;
    const RowChunks c(((c_i32_t)p.valid)[row_id], p.split);
    const int chunk = c.turned(p.by_chunks(id >> 3), qb);
    if (c.n > 1) {                         // sums of the chunk, relative to its maximum; combine_chunks_kernel goes on
      const size_t at = row_id * p.split.chunks + chunk;
      const float d_chunk = half_swap_sum_f32(dsum);
      uint32_t l = threadIdx.x & 63u;
      asm volatile("" : "+v"(l));
      const uint32_t q = wave * 32 + (l & 31u);
      float4 *const so = (float4 *)p.split.o + (at * 4 + wave) * (NDT * 4 * 64) + l;
#pragma unroll
      for (int i = 0; i < NDT * 4; i++)
        so[i * 64] = make_float4(O[i / 4][4 * (i % 4)], O[i / 4][4 * (i % 4) + 1], O[i / 4][4 * (i % 4) + 2], O[i / 4][4 * (i % 4) + 3]);
      if (l < 32) {
        p.split.md[at * 256 + q] = m;
        p.split.md[at * 256 + 128 + q] = d_chunk;
      }
      return;
    }
  }
  float dtot = half_swap_sum_f32(dsum);
  if constexpr (G > 1) {
    // the groups' sums, relative to the row's final maximum, meet in the (free) tile rings; group 0 goes on alone
    constexpr int GBYTES = 4 * 64 * NDT * 64;                // of one group's O
    static_assert((G - 1) * GBYTES <= (int)sizeof(smem), "O of the other groups fits the tile rings");
    const float f = __builtin_amdgcn_exp2f(m_own - m);
    dtot *= f;
#pragma unroll
    for (int dt = 0; dt < NDT; dt++)
#pragma unroll
      for (int e = 0; e < 16; e++) O[dt][e] *= f;
    __syncthreads();
    float4 *const so = (float4 *)smem + (wave * NDT * 4) * 64 + lane;
    if (grp > 0) {
      sFm[0][grp][wave * 32 + r] = dtot;
#pragma unroll
      for (int i = 0; i < NDT * 4; i++)
        so[(grp - 1) * (GBYTES / 16) + i * 64] = make_float4(O[i / 4][4 * (i % 4)], O[i / 4][4 * (i % 4) + 1], O[i / 4][4 * (i % 4) + 2], O[i / 4][4 * (i % 4) + 3]);
    }
    __syncthreads();
    if (grp == 0) {
#pragma unroll
      for (int g = 1; g < G; g++) {
        dtot += sFm[0][g][wave * 32 + r];
#pragma unroll
        for (int i = 0; i < NDT * 4; i++) {
          const float4 t = so[(g - 1) * (GBYTES / 16) + i * 64];
          O[i / 4][4 * (i % 4)] += t.x; O[i / 4][4 * (i % 4) + 1] += t.y; O[i / 4][4 * (i % 4) + 2] += t.z; O[i / 4][4 * (i % 4) + 3] += t.w;
        }
      }
    }
  }
  // (computed again: no register holds them across the loop)
  uint32_t lane_e = threadIdx.x & 63u;
  asm volatile("" : "+v"(lane_e));
  const float inv = __builtin_amdgcn_rcpf(dtot);
  // A lane holds four channels of one row per group: stored from here, an instruction would touch 32 rows with 16 bytes
  // each.  The rows of a wavefront go through LDS instead (the tile ring is free once every wavefront is past its last
  // P.V product) and leave as whole rows, 16 bytes per lane.
  constexpr int OROW = orow_bytes(D);
  static_assert(4 * 32 * OROW <= G * NBUF * (TILE + VTILE), "output rows of four wavefronts fit the tile ring");
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
  if (grp > 0) return;
  store_rows<D, ODT, PV16>(O, inv, smem + wave * (32 * OROW), sVscale, p, batch, head, qb * 128 + wave * 32, lane_e);
}

// ---- few short rows -------------------------------------------------------------------------------------------------
// A workgroup takes 32 QW queries of a row, a quarter or a half of it, and G wavefronts for each 32 of them, which take the row's blocks in
// turn, place rd G + grp of the list in round rd: several CUs to a row instead of one, and a row of up to G blocks in one round.
// Each wavefront has tiles of its own, and the next ones are requested as soon as the operands of the present ones are in registers;
// it meets the others once per round, to learn the running maximum in front of its block (P is rounded against it), and at the
// end, where O and the denominators are added up in the order of the groups.  No wavefront sees the votes of the row's other
// workgroups, so each skips a block on the vote of its own 32 queries: it skips whatever the whole row skips, whose V it then leaves
// alone, and at the thresholds of this route the rest as well adds nothing (few_rows).
// Arithmetic and masks are those of block_sparse_attn_kernel; at most 128 blocks to a row.
template <int D, int ODT, bool PV16, int SEL, int QW, int G>
__global__ __launch_bounds__(64 * QW * G, 2) void few_rows_attn_kernel(const AttnParams p) {
  constexpr int KS = D / 32, NDT = D / 32, TILE = 64 * D, VTILE = PV16 ? 2 * TILE : TILE, NKL = TILE / 1024, NVL = VTILE / 1024, W = SEL > 0 ? SEL : 1;
  constexpr int NI = NDT * 4, NW = QW * G, PARTS = 4 / QW;   // float4s of O per lane, wavefronts, workgroups to a row
  static_assert(NI * 1024 <= TILE + VTILE, "O of a wavefront fits its tiles");
  __shared__ __align__(1024) unsigned char smem[NW * (TILE + VTILE)];
  __shared__ float s_fm[2][G][QW * 32], s_d[G][QW * 32];
  __shared__ int s_ids[128];
  const int tid = threadIdx.x, lane = tid & 63, r = lane & 31, hh = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int grp = wave % G, qw = wave / G;
  int bh, qb;
  const int item = blockIdx.x, wg = (item >> 3) % PARTS;
  if (!place_workgroup(p, item & 7, (item >> 3) / PARTS, bh, qb)) return;
  const int first_row = qb * 128 + wg * (QW * 32), row0 = first_row + qw * 32;
  if (first_row >= p.N) return;
  const int batch = p.by_H(bh), head = bh - batch * p.H, bhk = batch * p.Hkv + p.by_group(head);
  const size_t row_id = (size_t)bh * p.nq + qb;
  const int Nk = p.Nk, last_col = p.nk - 1;
  if constexpr (!PV16) fp8_saturation_on();
  typedef const __attribute__((address_space(4))) int32_t *c_i32_t;
  typedef const __attribute__((address_space(4))) float *c_f32_t;
  const float qs = ((c_f32_t)p.q_scale)[p.q_per_warp ? row_id * 4 + wg * QW + qw : row_id];
  v4i qreg[KS];
#pragma unroll
  for (int ks = 0; ks < KS; ks++) {
    qreg[ks] = (v4i){0, 0, 0, 0};
    if (row0 + r < p.N) qreg[ks] = *(const v4i *)(p.q8 + ((size_t)bh * p.N + row0 + r) * D + 32 * ks + 16 * hh);
  }
  // the row's blocks, in a register each of places 0-63 and 64-127
  int nv, ids[2];
  if constexpr (SEL > 0) {
    __shared__ uint16_t s_score[64 * W];
    __shared__ int s_nv;
    const uint8_t *simk = p.sel.sim_k + (size_t)bhk * p.nk;
    const bool row_forced = p.sel.sim_q[row_id] == 0;
    bool k_dead[W];
#pragma unroll
    for (int t = 0; t < W; t++) k_dead[t] = simk[min(64 * t + lane, last_col)] == 0;
#pragma unroll
    for (int c0 = 0; c0 < 64 * W; c0 += 16 * NW) {
      const int col = c0 + (tid >> 2);
      if (64 * W % (16 * NW) == 0 || col < 64 * W) {
        const uint16_t s16 = pooled_score_4lanes<D, ODT>(p.sel.pool_q + row_id * D, p.sel.pool_k + ((size_t)bhk * p.nk + min(col, last_col)) * D, tid & 3);
        if ((tid & 3) == 0) s_score[col] = s16;
      }
    }
    __syncthreads();
    if (wave == 0) {
      const int causal_lim = p.sel.is_causal ? min(p.nk, 2 * (qb + 1)) : p.nk;
      uint64_t map[W] = {};
      float sc[W];
#pragma unroll
      for (int t = 0; t < W; t++) sc[t] = (64 * t + lane >= causal_lim || k_dead[t]) ? -INFINITY : elem_to_f32<ODT>(s_score[64 * t + lane]);
      select_row<ODT, W>(map, sc, k_dead, p.sel.by_topk, p.sel.level.at(head), p.nk, causal_lim, row_forced, p.sel.sink, lane);
      int before = 0;
#pragma unroll
      for (int t = 0; t < W; t++) {
        const int rank = before + __builtin_popcountll(map[t] & ((1ull << lane) - 1));
        if ((map[t] >> lane) & 1) s_ids[rank] = 64 * t + lane;
        before += __builtin_popcountll(map[t]);
      }
      if (lane == 0) s_nv = before;
    }
    __syncthreads();
    nv = __builtin_amdgcn_readfirstlane(s_nv);
    ids[0] = s_ids[lane];
    ids[1] = W > 1 ? s_ids[64 + lane] : 0;
    if (p.sel.valid_out != nullptr && tid == 0 && wg == 0) p.sel.valid_out[row_id] = nv;
  } else {
    nv = ((c_i32_t)p.valid)[row_id];
    const int32_t *list = p.lut + row_id * p.nk;
    const int d0 = list[min(lane, last_col)], d1 = list[min(64 + lane, last_col)];
    ids[0] = wave_prefix_sum(lane < nv ? d0 : 0);
    ids[1] = __builtin_amdgcn_readlane(ids[0], 63) + wave_prefix_sum(64 + lane < nv ? d1 : 0);
  }
  if (nv == 0) return;                                       // output rows stay unwritten (sm89.cuh:232-235)
  auto block_of = [&](int place) __attribute__((always_inline)) {
    return place < 64 ? __builtin_amdgcn_readlane(ids[0], place) : __builtin_amdgcn_readlane(ids[1], place - 64);
  };

  // tiles of this wavefront, laid out as block_sparse_attn_kernel has them
  typedef __attribute__((address_space(3))) void *lds_ptr_t;
  typedef const __attribute__((address_space(1))) void *glb_ptr_t;
  unsigned char *const sk = smem + wave * (TILE + VTILE), *const sv = sk + TILE;
  const uint32_t lds_k = (uint32_t)(size_t)(__attribute__((address_space(3))) unsigned char *)smem + (uint32_t)(wave * (TILE + VTILE)), lds_v = lds_k + TILE;
  const int8_t *kbase = p.k8 + (size_t)bhk * Nk * D;
  const uint8_t *vbase = p.v8 + (size_t)bhk * p.nk * (size_t)VTILE;
  const c_f32_t kscale = (c_f32_t)(p.k_scale + (size_t)bhk * p.nk);
  const uint32_t lane_off = ((uint32_t)lane ^ (D == 128 ? (lane >> 4) & 3u : (lane >> 4) & 1u)) << 4;
  auto load_k = [&](int b) __attribute__((always_inline)) {
    const int8_t *kb = kbase + (size_t)(uint32_t)b * TILE;
    const uint32_t last_row = (uint32_t)min(Nk - 1 - b * 64, 63);   // rows beyond Nk as that one: their scores are masked, their V rows are zero
#pragma unroll
    for (int u = 0; u < NKL; u++) {
      const uint32_t off = lane_off ^ (u >= NKL / 2 ? (D == 128 ? 64u : 32u) : 0u), row = (uint32_t)(u * (1024 / D)) + off / D;
      __builtin_amdgcn_global_load_lds((glb_ptr_t)(kb + min(row, last_row) * D + (off & (D - 1))), (lds_ptr_t)(sk + u * 1024), 16, 0, 0);
    }
  };
  auto load_v = [&](int b) __attribute__((always_inline)) {
    const uint8_t *vb = vbase + (size_t)(uint32_t)b * VTILE + lane * 16;
#pragma unroll
    for (int u = 0; u < NVL; u++) __builtin_amdgcn_global_load_lds((glb_ptr_t)(vb + u * 1024), (lds_ptr_t)(sv + u * 1024), 16, 0, 0);
  };
  int blk = block_of(min(grp, nv - 1));
  __builtin_amdgcn_s_waitcnt(0x0F70);                        // vmcnt(0): from here on it counts tiles only
  asm volatile("" ::: "memory");
  if (grp < nv) { load_k(blk); load_v(blk); }
  float ksc = kscale[blk];
  const int krow0 = 32 * ((r >> 2) & 1) + 4 * (r >> 3) + (r & 3), ksw = k_swz<D>(krow0);
  uint32_t kaddr[KS];
#pragma unroll
  for (int ks = 0; ks < KS; ks++) kaddr[ks] = lds_k + (uint32_t)(krow0 * D + ((hh ^ ksw) & 1) * 16) + ((uint32_t)(32 * ks) ^ (uint32_t)((ksw & 6) * 16));
  const uint32_t va_lo = lds_v + (uint32_t)(r * 64 + (((2 * hh) ^ v_swz(r)) * 16)), va_hi = va_lo ^ 16u;
  const uint32_t va16 = lds_v + (uint32_t)(r * 128 + (((4 * hh) ^ ((r >> 1) & 7)) * 16));
  const float thr = p.pvthr.p != nullptr ? ((c_f32_t)p.pvthr.p)[head] : p.pvthr.v;
  const float c = p.sm_scale_log2, cq26 = c * qs * SPG_ACC_SCALE, acc_c = __builtin_bit_cast(float, (int)SPG_ACC_C_BITS);
  const int kscale_precise_bits = __builtin_bit_cast(int, 16384.0f / (acc_c * cq26));
  float m = SPG_NEG_BIG, m_own = SPG_NEG_BIG, dsum = hh == 0 && grp == 0 ? 1.0f : 0.0f;
  v16f O[NDT];
#pragma unroll
  for (int dt = 0; dt < NDT; dt++)
#pragma unroll
    for (int e = 0; e < 16; e++) O[dt][e] = 0.f;
  const int rounds = (nv + G - 1) / G;
#pragma unroll 1
  for (int rd = 0; rd < rounds; rd++) {
    const int place = rd * G + grp;
    const bool active = place < nv, more = place + G < nv;
    float fm = -INFINITY, mloc = acc_c;
    const float dq = qs * ksc, a26 = cq26 * ksc;
    const bool precise = __builtin_bit_cast(int, ksc) >= kscale_precise_bits;
    int lim = 0x7fffffff, blk1 = blk;
    float ksc1 = ksc;
    bool masked = false;
    v16i S0, S1;
    if (active) {
      __builtin_amdgcn_s_waitcnt(0x0F70 | (NVL & 15) | ((NVL >> 4) << 14));   // K has arrived, V is under way
      asm volatile("" ::: "memory");
      v4i a0[KS], a1[KS];
      lds_read_4x128_wait<0, 16 * D>(a0[0], a1[0], a0[1], a1[1], kaddr[0], kaddr[1]);
      if constexpr (KS == 4) lds_read_4x128_wait<0, 16 * D>(a0[2], a1[2], a0[3], a1[3], kaddr[2], kaddr[3]);
      if (more) {
        blk1 = block_of(place + G);
        load_k(blk1);
        ksc1 = kscale[blk1];
      }
      asm volatile("v_mfma_i32_32x32x32_i8 %0, %2, %4, 0.15915494\n\tv_mfma_i32_32x32x32_i8 %1, %3, %4, 0.15915494"
                   : "=&v"(S0), "=&v"(S1)
                   : "v"(a0[0]), "v"(a1[0]), "v"(qreg[0]));
#pragma unroll
      for (int ks = 1; ks < KS; ks++) {
        S0 = __builtin_amdgcn_mfma_i32_32x32x32_i8(a0[ks], qreg[ks], S0, 0, 0, 0);
        S1 = __builtin_amdgcn_mfma_i32_32x32x32_i8(a1[ks], qreg[ks], S1, 0, 0, 0);
      }
      const int key0 = blk * 64 + 32 * hh;
      if (p.is_causal) lim = row0 + r - key0;                    // key > query (attn_utils.cuh:334-361)
      if (place == nv - 1) lim = min(lim, Nk - 1 - key0);        // key >= kv_len (attn_utils.cuh:363-389)
      masked = place >= nv - 2 && __any(lim < 31);
      if (!masked) {
        int imax = S0[0];
#pragma unroll
        for (int e = 1; e < 16; e++) imax = max(imax, S0[e]);
#pragma unroll
        for (int e = 0; e < 16; e++) imax = max(imax, S1[e]);
        mloc = __builtin_bit_cast(float, imax);
        fm = (mloc - acc_c) * a26;
      } else {
        fm = SPG_NEG_BIG;
        const float dq26 = dq * SPG_ACC_SCALE;
#pragma unroll
        for (int e = 0; e < 32; e++) {
          float v = (__builtin_bit_cast(float, e < 16 ? S0[e] : S1[e - 16]) - acc_c) * dq26;
          v = e > lim ? SPG_NEG_BIG : v;
          fm = fmaxf(fm, v);
        }
        fm = fm * c;
      }
      fm = half_swap_max_raw(fm);
    }
    s_fm[rd & 1][grp][qw * 32 + r] = fm;                         // (both halves hold the same value)
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    float before = m, after = -INFINITY, fms[G];
    lds_read_column<QW * 32>(fms, (uint32_t)(size_t)(__attribute__((address_space(3))) float *)&s_fm[rd & 1][0][qw * 32 + r]);
#pragma unroll
    for (int g = 0; g < G; g++) {
      if (g < grp) before = max_raw(before, fms[g]);
      if (g > grp) after = max_raw(after, fms[g]);
    }
    const float m_old = m_own, m_new = max_raw(before, fm);
    m = max_raw(m_new, after);
    if (active) {
      m_own = m_new;
      if (m_new > m_old) {
        const float osc = __builtin_amdgcn_exp2f(m_old - m_new);
        dsum *= osc;
#pragma unroll
        for (int dt = 0; dt < NDT; dt++)
#pragma unroll
          for (int e = 0; e < 16; e++) O[dt][e] *= osc;
      }
      // (All scores not a number: skipped, as in block_sparse_attn_kernel.  Only what V and P enter is left out: a branch in front of the exponentials
      // waits for the vote, one head N8192 D64 30.8 us per call without, 31.1 so, 32.0 with it there.)
      const bool skip = place < nv - 2 && !__any(fm - before + thr > 0.f);
      const float neg0 = PV16 ? -m_new : -m_new + SPG_FP8_OFFSET;
      float x[32];
      if (!masked) {
        float neg = __builtin_fmaf(-acc_c, a26, neg0), base = 0.f;
        if (__builtin_expect(precise, 0)) { neg = __builtin_fmaf(mloc - acc_c, a26, neg0); base = mloc; }   // (x - 0 is x)
#pragma unroll
        for (int e = 0; e < 32; e++) x[e] = __builtin_fmaf(__builtin_bit_cast(float, e < 16 ? S0[e] : S1[e - 16]) - base, a26, neg);
      } else {
        const float out = __builtin_fmaf(SPG_NEG_BIG, c, neg0), dq26 = dq * SPG_ACC_SCALE;
#pragma unroll
        for (int e = 0; e < 32; e++) {
          const float t = __builtin_fmaf((__builtin_bit_cast(float, e < 16 ? S0[e] : S1[e - 16]) - acc_c) * dq26, c, neg0);
          x[e] = e > lim ? out : t;
        }
      }
#pragma unroll
      for (int e = 0; e < 32; e++) x[e] = __builtin_amdgcn_exp2f(x[e]);
      // V: behind it only the next K may be under way
      if (more) __builtin_amdgcn_s_waitcnt(0x0F70 | (NKL & 15) | ((NKL >> 4) << 14));
      else __builtin_amdgcn_s_waitcnt(0x0F70);
      asm volatile("" ::: "memory");
      if constexpr (PV16) {
        typedef _Float16 h8 __attribute__((ext_vector_type(8)));
        typedef _Float16 h2 __attribute__((ext_vector_type(2)));
        typedef float f2 __attribute__((ext_vector_type(2)));
        h8 pb16[4];
        const h2 ones2 = {(_Float16)1, (_Float16)1};
        float rs = 0.f;
#pragma unroll
        for (int s4 = 0; s4 < 4; s4++)
#pragma unroll
          for (int j = 0; j < 8; j += 2) {
            const f2 pr = {x[8 * s4 + j], x[8 * s4 + j + 1]};
            const h2 ph = __builtin_convertvector(pr, h2);
            pb16[s4][j] = ph[0];
            pb16[s4][j + 1] = ph[1];
            rs = __builtin_amdgcn_fdot2(ph, ones2, rs, false);
          }
        if (!skip) {
          dsum += rs;
          v4i t[4][NDT];
#pragma unroll
          for (int st = 0; st < 4; st++) {
            const uint32_t a_ = va16 ^ (uint32_t)(16 * st);
            if constexpr (NDT == 4) { lds_read_4x128<0, 4096, 8192, 12288>(t[st][0], t[st][1], t[st][2], t[st][3], a_); lds_wait4(t[st][0], t[st][1], t[st][2], t[st][3]); }
            else { lds_read_2x128<0, 4096>(t[st][0], t[st][1], a_); lds_wait2(t[st][0], t[st][1]); }
#pragma unroll
            for (int dt = 0; dt < NDT; dt++)
              O[dt] = __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(h8, t[st][dt]), pb16[st], O[dt], 0, 0, 0);
          }
        }
        if (more) load_v(blk1);
      } else {
        float ps = x[0];
        if constexpr (D == 64) {
          // (the sums of block_sparse_attn_kernel)
          float pc[4] = {x[0], x[1], x[2], x[3]};
#pragma unroll
          for (int e = 4; e < 32; e++) pc[e % 4] += x[e];
          ps = (pc[0] + pc[1]) + (pc[2] + pc[3]);
        } else {
#pragma unroll
          for (int e = 1; e < 32; e++) ps += x[e];
        }
        v8i pb;
#pragma unroll
        for (int u = 0; u < 8; u++) pb[u] = pack4_e4m3(x[4 * u], x[4 * u + 1], x[4 * u + 2], x[4 * u + 3]);
        v4i lo[NDT], hi[NDT];
        if constexpr (NDT == 4) {
          lds_read_4x128_wait<0, 2048>(lo[0], lo[1], hi[0], hi[1], va_lo, va_hi);
          lds_read_4x128_wait<4096, 6144>(lo[2], lo[3], hi[2], hi[3], va_lo, va_hi);
        } else {
          lds_read_4x128_wait<0, 2048>(lo[0], lo[1], hi[0], hi[1], va_lo, va_hi);
        }
        if (more) load_v(blk1);
        if (!skip) {
          dsum += ps;
#pragma unroll
          for (int dt = 0; dt < NDT; dt++) {
            const v8i av = {lo[dt][0], lo[dt][1], lo[dt][2], lo[dt][3], hi[dt][0], hi[dt][1], hi[dt][2], hi[dt][3]};
            O[dt] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(av, pb, O[dt], 0, 0, 0, 0, 0, 0);
          }
        }
      }
    }
    blk = blk1;
    ksc = ksc1;
  }
  // the groups' sums, relative to the row's maximum, through their own tiles; group g then adds up float4s g, g + G, ... of the lanes
  const float f = __builtin_amdgcn_exp2f(m_own - m), d_own = half_swap_sum_f32(dsum) * f;
  if (hh == 0) s_d[grp][qw * 32 + r] = d_own;
  constexpr int SLOT = (TILE + VTILE) / 16;
  float4 *const so = (float4 *)smem + qw * (G * SLOT) + lane;
#pragma unroll
  for (int i = 0; i < NI; i++)
    so[grp * SLOT + i * 64] = make_float4(O[i / 4][4 * (i % 4)] * f, O[i / 4][4 * (i % 4) + 1] * f, O[i / 4][4 * (i % 4) + 2] * f, O[i / 4][4 * (i % 4) + 3] * f);
  float4 vsc[(NI + G - 1) / G];                              // V scales of the channels that this thread stores
#pragma unroll
  for (int u = 0; u < (NI + G - 1) / G; u++) {
    const int i = grp + u * G, d0 = 32 * (i / 4) + 8 * (i % 4) + 4 * hh;
    vsc[u] = make_float4(1.f, 1.f, 1.f, 1.f);
    if constexpr (!PV16) vsc[u] = *(const float4 *)(p.v_scale + (size_t)bhk * D + min(d0, D - 4));
  }
  __syncthreads();
  float d = s_d[0][qw * 32 + r];
#pragma unroll
  for (int g = 1; g < G; g++) d += s_d[g][qw * 32 + r];
  const float inv = __builtin_amdgcn_rcpf(d);
  uint16_t *const out = (uint16_t *)p.out + (size_t)batch * p.os.sb + (size_t)head * p.os.sh + (size_t)(row0 + r) * p.os.sn;
#pragma unroll
  for (int u = 0; u < (NI + G - 1) / G; u++) {
    const int i = grp + u * G, d0 = 32 * (i / 4) + 8 * (i % 4) + 4 * hh;
    if (i >= NI) continue;
    float4 s = so[i * 64];
#pragma unroll
    for (int g = 1; g < G; g++) {
      const float4 t = so[g * SLOT + i * 64];
      s.x += t.x; s.y += t.y; s.z += t.z; s.w += t.w;
    }
    const uint16_t o0 = f32_to_elem<ODT>(s.x * inv * vsc[u].x), o1 = f32_to_elem<ODT>(s.y * inv * vsc[u].y);
    const uint16_t o2 = f32_to_elem<ODT>(s.z * inv * vsc[u].z), o3 = f32_to_elem<ODT>(s.w * inv * vsc[u].w);
    if (row0 + r < p.N) *(uint2 *)(out + d0) = make_uint2((uint32_t)o0 | ((uint32_t)o1 << 16), (uint32_t)o2 | ((uint32_t)o3 << 16));
  }
}

// ---- rows in chunks ------------------------------------------------------------------------------------------------
// Maxima of the chunks of a row but the last, per query, over the scores as block_sparse_attn_kernel sees them: its running maximum
// in front of a chunk is the largest of those before it, to the bit, since it takes the same products in binary32.
// A wavefront holds all 128 queries and takes every fourth block of the chunk, with a tile of its own in LDS: nothing is read twice and
// nothing waits for another wavefront until the end.  (Operands straight from memory, 32 rows to an instruction, are bound by the lines that
// those touch: 35 us instead of 27 for 15 400 blocks at D = 128.)  Bound by its chain - count, list, Q block, tiles - and the rounding up to
// whole workgroups per CU: the matrix instructions of those 15 400 blocks take 7 us.
template <int D>
__global__ __launch_bounds__(256, D == 64 ? 4 : 3) void row_maxima_kernel(const AttnParams p) {
  constexpr int KS = D / 32;
  __shared__ __align__(1024) unsigned char s_tile[4][64 * D];   // of one wavefront each
  __shared__ __align__(1024) unsigned char s_q[128 * D];
  __shared__ int s_id[256], s_sum[2][4];
  __shared__ float s_max[4][128];
  const int tid = threadIdx.x, lane = tid & 63, r = lane & 31, hh = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  int bh, qb, chunk;
  if (!place_part(p, blockIdx.x, bh, qb, chunk)) return;
  const int batch = p.by_H(bh), head = bh - batch * p.H, bhk = batch * p.Hkv + p.by_group(head);
  const size_t row_id = (size_t)bh * p.nq + qb;
  const RowChunks chunks(p.valid[row_id], p.split);
  if (chunk >= (int)chunks.n - 1) return;            // (the maximum of a row's last chunk is nobody's)
  const int begin = chunks.begin(chunk), total = chunks.begin(chunk + 1) - begin;
  const int32_t *const list = p.lut + row_id * p.nk;
  int before = 0;                                    // sum of the differences in front
#pragma unroll 4
  for (int i = tid; i < begin; i += 256) before += list[i];
  int diff = tid < total ? list[begin + tid] : 0;
  const int behind = list[begin + total];
  typedef __attribute__((address_space(3))) void *lds_ptr_t;
  typedef const __attribute__((address_space(1))) void *glb_ptr_t;
  {
    // Q block to LDS, rows beyond N as the last one: chunks of 16 bytes swizzled as a K tile's
    const int8_t *qb8 = p.q8 + ((size_t)bh * p.N + qb * 128) * D;
    constexpr int CPR = D / 16;
#pragma unroll
    for (int u = 0; u < D / 32; u++) {
      const uint32_t pos = (uint32_t)((wave * (D / 32) + u) * 64 + lane), row_ = pos / CPR, slot = pos % CPR;
      const uint32_t off = min(row_, (uint32_t)(p.N - 1 - qb * 128)) * D + (slot ^ k_swz<D>(row_ & 63)) * 16u;
      __builtin_amdgcn_global_load_lds((glb_ptr_t)(qb8 + off), (lds_ptr_t)(s_q + (wave * (D / 32) + u) * 1024), 16, 0, 0);
    }
  }
  float cq26[4], m[4];
#pragma unroll
  for (int s = 0; s < 4; s++) {
    cq26[s] = p.sm_scale_log2 * p.q_scale[p.q_per_warp ? row_id * 4 + s : row_id] * SPG_ACC_SCALE;
    m[s] = SPG_NEG_BIG;
  }
  // a tile to LDS, one wavefront on its own: chunks of 16 bytes swizzled as block_sparse_attn_kernel has them
  constexpr int TILE = 64 * D;
  const int8_t *kbase = p.k8 + (size_t)bhk * p.Nk * D;
  const uint32_t lane_off = ((uint32_t)lane ^ (D == 128 ? (lane >> 4) & 3u : (lane >> 4) & 1u)) << 4;
  unsigned char *const tile = s_tile[wave];
  auto fetch = [&](int blk) __attribute__((always_inline)) {
    const int8_t *kb = kbase + (size_t)(uint32_t)blk * TILE;
#pragma unroll
    for (int u = 0; u < TILE / 1024; u++)       // rows from 32 on: one more bit of the swizzle
      __builtin_amdgcn_global_load_lds((glb_ptr_t)(kb + u * 1024 + (lane_off ^ (u >= TILE / 2048 ? (D == 128 ? 64u : 32u) : 0u))),
                                       (lds_ptr_t)(tile + u * 1024), 16, 0, 0);
  };
  const int krow0 = 32 * ((r >> 2) & 1) + 4 * (r >> 3) + (r & 3), ksw = k_swz<D>(krow0);
  const uint32_t k_rd = (uint32_t)(size_t)(__attribute__((address_space(3))) unsigned char *)tile + (uint32_t)(krow0 * D + ((hh ^ ksw) & 1) * 16);
  uint32_t kaddr[KS];
#pragma unroll
  for (int ks = 0; ks < KS; ks++) kaddr[ks] = k_rd + ((uint32_t)(32 * ks) ^ (uint32_t)((ksw & 6) * 16));
  const float *kscale = p.k_scale + (size_t)bhk * p.nk;
  before = wave_prefix_sum(before);
  if (lane == 63) s_sum[1][wave] = before;
  int base = 0;
  v4i q[4][KS];
  for (int t0 = 0; t0 < total; t0 += 256) {
    // ids of up to 256 blocks: running sums of the differences
    const int n = min(256, total - t0);
    if (t0 > 0) diff = tid < n ? list[begin + t0 + tid] : 0;
    int s = wave_prefix_sum(diff);
    if (lane == 63) s_sum[0][wave] = s;
    __builtin_amdgcn_s_waitcnt(0x0F70);        // vmcnt(0): this wavefront's share of the Q block
    __syncthreads();
    if (t0 == 0) {
      base = s_sum[1][0] + s_sum[1][1] + s_sum[1][2] + s_sum[1][3];
#pragma unroll
      for (int s4 = 0; s4 < 4; s4++) {
        // query 32 s4 + r, chunk 2 ks + hh
#pragma unroll
        for (int ks = 0; ks < KS; ks++) {
          q[s4][ks] = *(const v4i *)(s_q + (32 * s4 + r) * D + (((2 * ks + hh) ^ k_swz<D>((32 * s4 + r) & 63)) * 16));
          if (qb * 128 + 32 * s4 + r >= p.N) q[s4][ks] = (v4i){0, 0, 0, 0};
        }
      }
    }
    s += base;
    for (int w = 0; w < wave; w++) s += s_sum[0][w];
    base += s_sum[0][0] + s_sum[0][1] + s_sum[0][2] + s_sum[0][3];
    s_id[tid] = s;
    __syncthreads();
    const int ids = s_id[min(wave + 4 * lane, n - 1)];         // of this wavefront: in a register
    const int mine = wave < n ? (n - wave + 3) / 4 : 0;
    int blk = __builtin_amdgcn_readlane(ids, 0);
    if (mine > 0) fetch(blk);
    float ksc = kscale[blk];
#pragma unroll 1
    for (int i = 0; i < mine; i++) {
      v4i a[2][KS];
      __builtin_amdgcn_s_waitcnt(0x0F70);      // vmcnt(0): the tile has arrived
      asm volatile("" ::: "memory");
      lds_read_4x128_wait<0, 16 * D>(a[0][0], a[1][0], a[0][1], a[1][1], kaddr[0], kaddr[1]);
      if constexpr (KS == 4) lds_read_4x128_wait<0, 16 * D>(a[0][2], a[1][2], a[0][3], a[1][3], kaddr[2], kaddr[3]);
      blk = __builtin_amdgcn_readlane(ids, min(i + 1, 63));
      if (i + 1 < mine) fetch(blk);            // under the products; the operands are in registers
      const float ksc1 = kscale[blk];
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int s4 = 0; s4 < 4; s4++) {
        v16i S0, S1;
        // (both chains beside each other: left to itself the compiler puts them one behind the other into the same registers)
        asm volatile("v_mfma_i32_32x32x32_i8 %0, %2, %4, 0\n\tv_mfma_i32_32x32x32_i8 %1, %3, %4, 0"
                     : "=&v"(S0), "=&v"(S1)
                     : "v"(a[0][0]), "v"(a[1][0]), "v"(q[s4][0]));
#pragma unroll
        for (int ks = 1; ks < KS; ks++) {
          S0 = __builtin_amdgcn_mfma_i32_32x32x32_i8(a[0][ks], q[s4][ks], S0, 0, 0, 0);
          S1 = __builtin_amdgcn_mfma_i32_32x32x32_i8(a[1][ks], q[s4][ks], S1, 0, 0, 0);
        }
        int imax = S0[0];
#pragma unroll
        for (int e = 1; e < 16; e++) imax = max(imax, S0[e]);
#pragma unroll
        for (int e = 0; e < 16; e++) imax = max(imax, S1[e]);
        // 2^-26 imax is what the attention kernel reads off its accumulator
        m[s4] = fmaxf(m[s4], ((float)imax * (1.0f / SPG_ACC_SCALE)) * (cq26[s4] * ksc));
      }
      ksc = ksc1;
    }
    __syncthreads();
  }
  if (tid == 0) p.split.first[row_id * p.split.chunks + chunk + 1] = base + behind;   // where the next chunk starts
#pragma unroll
  for (int s = 0; s < 4; s++) {
    const float v = half_swap_max_f32(m[s]);
    if (lane < 32) s_max[wave][s * 32 + r] = v;
  }
  __syncthreads();
  if (tid < 128)
    p.split.maxima[(row_id * p.split.chunks + chunk) * 128 + tid] = fmaxf(fmaxf(s_max[0][tid], s_max[1][tid]), fmaxf(s_max[2][tid], s_max[3][tid]));
}

// The chunks of a row, each relative to its own maximum, brought to the row's (that of the last chunk) and added up in their order.
// A workgroup takes 32 channels of a row, as the lanes of the attention kernel hold them.
template <int D, int ODT, bool PV16>
__global__ __launch_bounds__(256) void combine_chunks_kernel(const AttnParams p) {
  constexpr int NDT = D / 32;
  const int tid = threadIdx.x, lane = tid & 63, r = lane & 31, hh = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  int bh, qb, dt;
  if (!place_part(p, blockIdx.x, bh, qb, dt)) return;
  const int batch = p.by_H(bh), head = bh - batch * p.H, bhk = batch * p.Hkv + p.by_group(head);
  const size_t row_id = (size_t)bh * p.nq + qb;
  const int chunks = (int)RowChunks(p.valid[row_id], p.split).n;
  if (chunks == 1) return;                 // the row is finished
  const float *md = p.split.md + row_id * p.split.chunks * 256 + wave * 32 + r;
  const float4 *so = (const float4 *)p.split.o + (row_id * p.split.chunks * 4 + wave) * (NDT * 4 * 64) + dt * (4 * 64) + lane;
  const float m = md[(chunks - 1) * 256];
  float d = 0.f;
  float4 O[4];
#pragma unroll
  for (int g = 0; g < 4; g++) O[g] = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll 4
  for (int c = 0; c < chunks; c++) {
    const float f = __builtin_amdgcn_exp2f(md[c * 256] - m);
    d += md[c * 256 + 128] * f;
#pragma unroll
    for (int g = 0; g < 4; g++) {
      const float4 t = so[(size_t)c * (4 * NDT * 4 * 64) + g * 64];
      O[g].x += t.x * f; O[g].y += t.y * f; O[g].z += t.z * f; O[g].w += t.w * f;
    }
  }
  const float inv = __builtin_amdgcn_rcpf(d);
  const int q_row = qb * 128 + wave * 32 + r;
  if (q_row >= p.N) return;
  uint16_t *const out = (uint16_t *)p.out + (size_t)batch * p.os.sb + (size_t)head * p.os.sh + (size_t)q_row * p.os.sn;
#pragma unroll
  for (int g = 0; g < 4; g++) {
    const int d0 = 32 * dt + 8 * g + 4 * hh;
    float4 sc = make_float4(1.f, 1.f, 1.f, 1.f);
    if constexpr (!PV16) sc = *(const float4 *)(p.v_scale + (size_t)bhk * D + d0);
    const uint16_t o0 = f32_to_elem<ODT>(O[g].x * inv * sc.x), o1 = f32_to_elem<ODT>(O[g].y * inv * sc.y);
    const uint16_t o2 = f32_to_elem<ODT>(O[g].z * inv * sc.z), o3 = f32_to_elem<ODT>(O[g].w * inv * sc.w);
    *(uint2 *)(out + d0) = make_uint2((uint32_t)o0 | ((uint32_t)o1 << 16), (uint32_t)o2 | ((uint32_t)o3 << 16));
  }
}

// Few long rows: each over several workgroups (rows_in_chunks has the line).  One workgroup per row leaves CUs idle, ends when the longest
// row ends, and has its groups of wavefronts meet at a barrier for every round of blocks; what stands against cutting the row is that P is
// rounded against the running maximum.  Scores and maxima alone need no order and are a third of the work: a launch in front takes the maxima of
// the chunks, after which the chunks are independent.  One head N17776 D64 with every block kept: 133 us in groups; 24 + 78 + 11 in chunks.
template <int D, int ODT, bool PV16>
static void launch_split(AttnParams &p, hipStream_t st) {
  const int per_xcd = (p.total_wg + 7) / 8;
  p.split.rows = p.total_wg;
  p.by_chunks = FastDiv::of(per_xcd);
  row_maxima_kernel<D><<<8 * per_xcd * (p.split.chunks - 1), 256, 0, st>>>(p);
  block_sparse_attn_kernel<D, ODT, PV16, 0, 1, 0, true><<<8 * per_xcd * p.split.chunks, 256, 0, st>>>(p);
  combine_chunks_kernel<D, ODT, PV16><<<8 * per_xcd * (D / 32), 256, 0, st>>>(p);
}

template <int SEL, int FQ>
static hipError_t launch_attn(AttnParams &p, int D, int out_dtype, bool causal_rows, hipStream_t st) {
  p.nq = (p.N + 127) / 128; p.nk = (p.Nk + 63) / 64;
  p.total_wg = p.nq * p.H * p.B;
  p.wg_per_xcd = (p.total_wg + 7) / 8;
  // The queue costs a row an atomic round trip before it can start and gains it a share of its time: it takes rows long enough,
  // and several rounds of them.  A row is nk blocks of D channels, half of that on average where the selection is causal.  us per
  // call with / without, N or H x N, top-k 0.3 to 0.5: D64 96 x 6000 450 / 431, 32 x 16384 941 / 932, 24 x 16448 677 / 677, 23 x 17000
  // 789 / 796, 48 x 32768 5095 / 5180; D128 96 x 6000 659 / 652, 96 x 8192 1046 / 1051, 48 x 12288 1047 / 1060; causal D64 40 x 16384
  // 976 / 952, 32 x 32768 2681 / 2670, 28 x 40000 3755 / 3755, 12 x 65536 4334 / 4422; causal D128 96 x 8192 1057 / 1043, 32 x 16384
  // 1138 / 1134, 48 x 24576 3624 / 3650, 12 x 65536 6161 / 6330, 11 x 90000 10188 / 10864.  Fewer rows per XCD: D64 8 x 16384 278 / 269,
  // 20 x 16384 628 / 618, 18 x 17000 647 / 641, D128 8 x 16384 396 / 389, 18 x 17000 894 / 901; causal D128 18 x 17000 724 / 714.
  const long long row = ((long long)p.nk * D) >> (causal_rows ? 1 : 0);
  if (SEL > 0 || p.wg_per_xcd < SPG_QUEUE_MIN || row <= SPG_QUEUE_MIN_ROW) p.queue = nullptr;
  const int grid = 8 * (p.queue != nullptr ? p.wg_per_xcd + p.wg_per_xcd / SPG_QUEUE_EXTRA : p.wg_per_xcd);
  // Causal rows differ in length throughout: all rows by length while the heads an XCD works on at once share its L2
  // anyway (grids of a few rounds), head by head beyond.  Otherwise only a partial last Q block stands out.
  p.rows_first = (causal_rows && p.wg_per_xcd <= SPG_ROW_MAJOR_MAX) ? p.nq : (p.N % 128 != 0 || causal_rows) ? 1 : 0;
  p.by_nq = FastDiv::of(p.nq); p.by_rest = FastDiv::of(p.nq > p.rows_first ? p.nq - p.rows_first : 1);
  p.by_H = FastDiv::of(p.H); p.by_group = FastDiv::of(p.H / p.Hkv);
  if constexpr (FQ == 0) {
    if (p.few > 0) {
      p.queue = nullptr;
#define SPG_FEW_(D_, PV16_, QW_, G_)                                                                                        \
  {                                                                                                                         \
    const int wgs = 8 * (4 / QW_) * p.wg_per_xcd;                                                                           \
    if (out_dtype == 0) few_rows_attn_kernel<D_, 0, PV16_, SEL, QW_, G_><<<wgs, 64 * QW_ * G_, 0, st>>>(p);                    \
    else few_rows_attn_kernel<D_, 1, PV16_, SEL, QW_, G_><<<wgs, 64 * QW_ * G_, 0, st>>>(p);                                   \
  }
#define SPG_FEW(D_, PV16_, NW_) { if (p.few == 4) SPG_FEW_(D_, PV16_, 1, NW_) else SPG_FEW_(D_, PV16_, 2, NW_ / 2) }
      // (the FP16 tiles of eight wavefronts at D = 128 would not fit the LDS)
      if (p.v_scale != nullptr) { if (D == 64) SPG_FEW(64, false, 8) else SPG_FEW(128, false, 8) }
      else { if (D == 64) SPG_FEW(64, true, 8) else SPG_FEW_(128, true, 1, 6) }
#undef SPG_FEW
#undef SPG_FEW_
      return hipGetLastError();
    }
  }
  if constexpr (SEL == 0 && FQ == 0) {
    if (p.split.chunks > 1) {
      p.queue = nullptr;
#define SPG_SPLIT(D_, PV16_) { if (out_dtype == 0) launch_split<D_, 0, PV16_>(p, st); else launch_split<D_, 1, PV16_>(p, st); }
      if (p.v_scale != nullptr) { if (D == 64) SPG_SPLIT(64, false) else SPG_SPLIT(128, false) }
      else { if (D == 64) SPG_SPLIT(64, true) else SPG_SPLIT(128, true) }
#undef SPG_SPLIT
      return hipGetLastError();
    }
  }
  const int n_groups = FQ == 0 && p.pv_mode == 1 && p.pv_count == nullptr ? attn_groups(p.total_wg, p.nk, D, p.v_scale == nullptr) : 1;
#define SPG_ATTN(D_, PV16_, G_)                                                                             \
  {                                                                                                         \
    if (out_dtype == 0) block_sparse_attn_kernel<D_, 0, PV16_, SEL, G_, FQ, false><<<grid, 256 * G_, 0, st>>>(p);  \
    else block_sparse_attn_kernel<D_, 1, PV16_, SEL, G_, FQ, false><<<grid, 256 * G_, 0, st>>>(p);                 \
  }
#define SPG_ATTN_G(D_, PV16_)                                                                               \
  {                                                                                                         \
    constexpr int GMAX = SEL == 1 ? 2 : D_ == 64 ? 4 : PV16_ ? 2 : 3;                                              \
    if constexpr (FQ > 0) {                                                                                 \
      if constexpr (D_ == 128) SPG_ATTN(D_, PV16_, 1)                                                        \
      else return hipErrorInvalidValue;                                                                     \
    } else if (n_groups == 1) SPG_ATTN(D_, PV16_, 1)                                                         \
    else if (n_groups == 2) SPG_ATTN(D_, PV16_, 2)                                                           \
    else if constexpr (GMAX > 2) SPG_ATTN(D_, PV16_, GMAX)                                                   \
  }
  if (p.v_scale != nullptr) { if (D == 64) SPG_ATTN_G(64, false) else SPG_ATTN_G(128, false) }
  else { if (D == 64) SPG_ATTN_G(64, true) else SPG_ATTN_G(128, true) }   // fp16 V^T tiles, no V scale
#undef SPG_ATTN_G
#undef SPG_ATTN
  return hipGetLastError();
}

hipError_t launch_block_sparse_attn_h(const int8_t *q8, const int8_t *k8, const uint8_t *v8, void *out, Strides os,
                                      int out_dtype, const int32_t *lut, const int32_t *valid, const RowSelect *sel, const RawQ *q,
                                      Hyper pvthreshd, const float *q_scale, const float *k_scale, const float *v_scale,
                                      int B, int H, int Hkv, int N, int Nk, int D, float sm_scale, int is_causal,
                                      int q_per_warp, int pv_mode, int32_t *pv_count, bool causal_rows, int *queue, const RowSplit *split, int few,
                                      hipStream_t st) {
  AttnParams p = {};
  p.queue = queue;
  p.few = few;
  if (split != nullptr) p.split = *split;
  p.q8 = q8; p.k8 = k8; p.v8 = v8; p.out = out; p.os = os; p.lut = lut; p.valid = valid; p.pvthr = pvthreshd;
  p.q_scale = q_scale; p.k_scale = k_scale; p.v_scale = v_scale; p.pv_count = pv_count;
  p.B = B; p.H = H; p.Hkv = Hkv; p.N = N; p.Nk = Nk;
  p.sm_scale_log2 = sm_scale * SPG_LOG2E;
  p.is_causal = is_causal;
  p.pv_mode = pv_mode;
  p.q_per_warp = q_per_warp;
  if (q != nullptr) p.q = *q;
  const bool causal = causal_rows || is_causal;
  if (sel == nullptr) return q != nullptr ? launch_attn<0, 1>(p, D, out_dtype, causal, st) : launch_attn<0, 0>(p, D, out_dtype, causal, st);
  p.sel = *sel;
  if (Nk <= 64 * 64) return q != nullptr ? launch_attn<1, 2>(p, D, out_dtype, causal, st) : launch_attn<1, 0>(p, D, out_dtype, causal, st);
  return q != nullptr ? launch_attn<2, 2>(p, D, out_dtype, causal, st) : launch_attn<2, 0>(p, D, out_dtype, causal, st);
}

hipError_t launch_block_sparse_attn(const int8_t *q8, const int8_t *k8, const uint8_t *v8, void *out, Strides os,
                                    int out_dtype, const int32_t *lut, const int32_t *valid, const float *pvthreshd,
                                    const float *q_scale, const float *k_scale, const float *v_scale, int B, int H,
                                    int Hkv, int N, int Nk, int D, float sm_scale, int is_causal, int q_per_warp,
                                    int pv_mode, int32_t *pv_count, hipStream_t st) {
  return launch_block_sparse_attn_h(q8, k8, v8, out, os, out_dtype, lut, valid, nullptr, nullptr, Hyper{pvthreshd, 0.f}, q_scale, k_scale,
                                    v_scale, B, H, Hkv, N, Nk, D, sm_scale, is_causal, q_per_warp, pv_mode, pv_count, false, nullptr, nullptr, 0, st);
}

}  // namespace spg
