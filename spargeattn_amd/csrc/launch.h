// Host-side launch functions shared between the kernel translation units and the C ABI (capi.hip).
#pragma once
#include <hip/hip_runtime.h>
#include <stddef.h>
#include <stdint.h>

namespace spg {

// Element strides of a (B, H, N, D) tensor whose last dimension is contiguous: element (b, h, n, d) sits at
// b*sb + h*sh + n*sn + d.  HND-contiguous: {H*N*D, N*D, D}; NHD-contiguous (B, N, H, D in memory): {N*H*D, D, H*D}.
struct Strides {
  long long sb, sh, sn;
};

// A per-head hyper-parameter: (H,) values on the device, or one value for all heads.  The second form takes no device
// memory and no fill kernel.
struct Hyper {
  const float *p;
  float v;
#ifdef __HIPCC__
  __device__ float at(int h) const { return p != nullptr ? p[h] : v; }
#endif
};

size_t km_mean_workspace_bytes(int B, int H, int N, int D);
void launch_km_mean(const void *k, Strides ks, void *km, void *ws, int B, int H, int N, int D, int dtype, hipStream_t st);
// size of the library-owned scratch array behind launch_km_mean_static (bytes); a shape whose
// km_mean_workspace_bytes() exceeds it is refused by the caller
#define SPG_KM_STATIC_SCRATCH_BYTES (8u << 20)
size_t km_mean_static_capacity();
hipError_t launch_km_mean_static(const void *k, Strides ks, void *km, int B, int H, int N, int D, int dtype, hipStream_t st);
void launch_pool_sim_quant(const void *x, Strides xs, const void *km, void *pool, uint8_t *sim, int8_t *xq, float *scale,
                           const float *thr, int B, int H, int N, int D, int block, int quant_rows, int dtype,
                           hipStream_t st);
int block_select_max_nk();
hipError_t launch_block_select(const void *pq, const uint8_t *sq, const void *pk, const uint8_t *sk, const float *topk,
                               const float *cdf, int causal, int sink, int32_t *lut, int32_t *valid, uint8_t *bmap,
                               int B, int H, int Hkv, int nq, int nk, int D, int dtype, hipStream_t st);
// the same with the level (top-k fraction or CDF threshold) as a Hyper; valid_out: the counts once more, where the host can see them, or NULL
hipError_t launch_block_select_h(const void *pq, const uint8_t *sq, const void *pk, const uint8_t *sk, bool by_topk,
                                 Hyper level, int causal, int sink, int32_t *lut, int32_t *valid, int32_t *valid_out, uint8_t *bmap,
                                 int B, int H, int Hkv, int nq, int nk, int D, int dtype, hipStream_t st);
void launch_div_selftest(unsigned long long *counts, int n_div, uint32_t seed, hipStream_t st);
hipError_t launch_map_to_lut(const void *mask, int kind, int32_t *lut, int32_t *valid, int B, int H, int nq, int nk,
                             hipStream_t st);

void launch_v_quant_fp8(const void *v, Strides vs, uint8_t *v8, float *v_scale, int B, int H, int N, int D, int dtype,
                        hipStream_t st);

void launch_v_tiles_f16(const void *v, Strides vs, void *vt, int B, int H, int N, int D, int dtype, hipStream_t st);

hipError_t launch_block_sparse_attn(const int8_t *q8, const int8_t *k8, const uint8_t *v8, void *out, Strides os,
                                    int out_dtype,
                                    const int32_t *lut, const int32_t *valid, const float *pvthreshd,
                                    const float *q_scale, const float *k_scale, const float *v_scale, int B, int H,
                                    int Hkv, int N, int Nk, int D, float sm_scale, int is_causal, int q_per_warp,
                                    int pv_mode, int32_t *pv_count, hipStream_t st);
// What the attention kernel needs to select a row's blocks by itself (rows of at most SPG_SELECT_IN_ATTN_NK blocks):
// the arguments of launch_block_select_h.  us per call with a selection kernel / in place, 65 to 128 blocks: D128 H1 N8192 76.6 / 71.1,
// H8 127.3 / 120.5, H24 310 / 305, FP16 PV H24 causal 326 / 320, CDF H20 N7000 386 / 381; D64 H4 62.4 / 59.2, H40 337.5 / 337.8.  129 to
// 256 blocks would gain at D128 (H8 N9000 190.3 / 186.7, H1 119.0 / 119.6) and lose at D64 (H2 N16384 95.8 / 105.4, H20 N16000 570 / 580),
// FP16 PV (H10 N12000 380 / 387) and on long grids (H16 N16000 671 / 679).
#define SPG_SELECT_IN_ATTN_NK 128
struct RowSelect {
  const uint16_t *pool_q, *pool_k;
  const uint8_t *sim_q, *sim_k;
  Hyper level;
  int by_topk, is_causal, sink;
  int32_t *valid_out;               // counts for the caller, or NULL
};
// Q as the caller has it, for an attention kernel that quantises it (and pools it, with a RowSelect) in place: one scale per block or per 32 rows
// as q_per_warp says, simthr as psq_core takes it.
struct RawQ {
  const uint16_t *x;
  Strides st;
  Hyper simthr;
};
// Groups of wavefronts per row (attn.hip, template argument G).  A row alone on its CU: its blocks go over groups.  As many groups
// as registers and LDS allow where rows are long, two for shorter ones, where the exchange and the final sum weigh more.  us per call
// with 1 / 2 / 3 / 4 groups, D64: one head N17776 281 / 236 / 169 / 163.5 (the last two of a later build), H2 N16384 131 / 111 / 98.4 / 96.2, H2
// N12000 CDF - / - / 123.5 / 120.7; H8 N4096 45 / 39.2 / 39.0 / 39.8, H2 N2048 - / 25.8 / 26.3 / 27.2; H2 N256 18.0 / 18.6 / 19.9.  D128: one head
// N17776 - / 227 / 214, H2 N16384 161 / 131 / 127, H2 N12000 causal - / 166 / 157.5; H8 N4096 59 / 53.5 / 54.0, H4 N3584 - / 42.4 / 43.1, H2
// N2304 - / 32.6 / 33.4, H2 N1024 - / 25.2 / 26.6.  FP16 PV D128 H2 N16384 188 / 164 (two fit the LDS).
// D128 with two / three groups around the line: rows that keep all blocks (the partial last row of a head does) H2 N4500 69.0 / 67.5,
// H2 N6100 90.6 / 88.4, one head 130 x 4200 60.6 / 59.3, 500 x 6100 87.8 / 85.6; whole rows with top-k 0.3 and 0.6 lose a little or gain: H2
// N5120 41.0 / 42.4 and 57.4 / 57.6, N6144 46.7 / 48.2 and 66.7 / 65.8, 8 rows of Nk 6144 51.9 / 53.0 and 72.8 / 71.8.  The number of rows
// makes no difference: one row of Nk 17776 134.1 / 128.4, 32768 216 / 205, 300000 1781 / 1659; 4 rows of 8200 73.8 / 71.5, 7 rows of 12000 98.5 / 95.0.
// Beyond one row per CU the rows fill each other's gaps: H10 N4096 unchanged without groups.  Lists of the caller's own in a head
// longer than the operators take (32768 blocks) say nothing of their length by nk: two, as over a short head.
inline int attn_groups(int rows, int nk, int D, bool pv_f16) {
  if (rows > 256 || nk < 12) return 1;
  if (nk <= 64) return 2;
  return D == 64 ? 4 : !pv_f16 && nk <= 32768 ? 3 : 2;
}
// A row's blocks over several workgroups, and scratch for what these leave behind.
struct RowSplit {
  int chunks;                       // workgroups of a row at most; 0 or 1: one
  int per;                          // blocks of a workgroup at most
  int rows;                         // (set at the launch)
  int *first;                       // [rows][chunks]            first block of a chunk
  float *maxima;                    // [rows][chunks][128]       largest score of a chunk
  float *md;                        // [rows][chunks][2][128]    running maximum at its end, denominator
  float *o;                         // [rows][chunks][128 x D]   sums, as the lanes hold them
};
// few: workgroups to a row as few_rows (forward_plan.h) has them, with q == NULL and pv_count == NULL, or 0.
// split: with sel == NULL, q == NULL, pv_count == NULL and the per-block PV threshold only.
// sel == NULL: blocks come from lut / valid; otherwise they are selected in place and lut / valid are not read.
// q == NULL: Q comes as q8 / q_scale (and pooled in sel); otherwise from the caller's tensor, and those are not read.
// queue: 8 device ints, zero when the kernel starts, for handing out rows across the XCDs, or NULL for a fixed share each.
// causal_rows: the selection is causal, so rows get longer with their index (order of the workgroups only).
hipError_t launch_block_sparse_attn_h(const int8_t *q8, const int8_t *k8, const uint8_t *v8, void *out, Strides os,
                                      int out_dtype, const int32_t *lut, const int32_t *valid, const RowSelect *sel, const RawQ *q,
                                      Hyper pvthreshd, const float *q_scale, const float *k_scale, const float *v_scale,
                                      int B, int H, int Hkv, int N, int Nk, int D, float sm_scale, int is_causal,
                                      int q_per_warp, int pv_mode, int32_t *pv_count, bool causal_rows, int *queue,
                                      const RowSplit *split, int few, hipStream_t st);
void launch_fp8_pack_selftest(const float *x, uint8_t *codes, int n, int saturate, hipStream_t st);

hipError_t launch_dense_attn_f16(const void *q, const void *k, const void *v, void *out, int B, int H, int N, int D,
                                 float sm_scale, int is_causal, hipStream_t st);

}  // namespace spg
