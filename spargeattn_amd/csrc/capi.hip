// extern "C" entry points declared in include/spargeattn_amd.h: argument checks, then a launch on the caller's
// stream.  No allocation, no synchronisation; the only state is the thread-local error string and, behind
// spg_km_mean_static, a library-owned device array per GPU with its cached address.
#include "capi_checks.h"
#include "forward_plan.h"

#include <chrono>
#include <cmath>
#include <cstdarg>
#include <cstdio>
#include <thread>

static thread_local char g_err[512] = "";

namespace spg {
int fail(int code, const char *fmt, ...) {
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(g_err, sizeof(g_err), fmt, ap);
  va_end(ap);
  return code;
}
}  // namespace spg
using namespace spg;

extern "C" {

int spg_version(void) { return 100; }

const char *spg_last_error(void) { return g_err; }

size_t spg_km_mean_workspace_bytes(int B, int H, int N, int D) {
  if (B <= 0 || H <= 0 || N <= 0 || D <= 0) return 0;
  return spg::km_mean_workspace_bytes(B, H, N, D);
}

int spg_km_mean(const void *k, const int64_t *k_strides, void *km, void *workspace, int B, int H, int N, int D, int dtype, void *stream) {
  const char *fn = "spg_km_mean";
  SPG_TRY(check_shape(fn, B, H, N, D));
  SPG_TRY(check_dtype(fn, dtype));
  SPG_NONNULL(fn, k); SPG_NONNULL(fn, km); SPG_NONNULL(fn, workspace);
  spg::Strides ks;
  SPG_TRY(get_strides(fn, "k_strides", k_strides, H, N, D, &ks));
  spg::launch_km_mean(k, ks, km, workspace, B, H, N, D, dtype, (hipStream_t)stream);
  return check_launch(fn, hipSuccess);
}

int spg_km_mean_static(const void *k, const int64_t *k_strides, void *km, int B, int H, int N, int D, int dtype, void *stream) {
  const char *fn = "spg_km_mean_static";
  SPG_TRY(check_shape(fn, B, H, N, D));
  SPG_TRY(check_dtype(fn, dtype));
  SPG_NONNULL(fn, k); SPG_NONNULL(fn, km);
  const size_t need = spg::km_mean_workspace_bytes(B, H, N, D);
  if (need > spg::km_mean_static_capacity())
    return fail(SPG_ERR_UNSUPPORTED, "%s: B=%d H=%d N=%d D=%d needs %zu bytes of scratch, the built-in array holds %zu "
                "(use spg_km_mean with a workspace of your own)", fn, B, H, N, D, need, spg::km_mean_static_capacity());
  spg::Strides ks;
  SPG_TRY(get_strides(fn, "k_strides", k_strides, H, N, D, &ks));
  const hipError_t e = spg::launch_km_mean_static(k, ks, km, B, H, N, D, dtype, (hipStream_t)stream);
  if (e == hipErrorInvalidDevice)
    return fail(SPG_ERR_INVALID, "%s: the stream's device must be the current device (the built-in array is per GPU)", fn);
  return check_launch(fn, e);
}

int spg_pool_sim_quant(const void *x, const int64_t *x_strides, const void *km, void *pool, uint8_t *sim, int8_t *xq, float *scale,
                       const float *simthreshd1, int B, int H, int N, int D, int block, int quant_rows, int dtype, void *stream) {
  const char *fn = "spg_pool_sim_quant";
  SPG_TRY(check_shape(fn, B, H, N, D));
  SPG_TRY(check_dtype(fn, dtype));
  if (block != 64 && block != 128) return fail(SPG_ERR_UNSUPPORTED, "%s: block must be 64 or 128 (got %d)", fn, block);
  if (quant_rows != block && !(quant_rows == 32 && block == 128 && km == nullptr))
    return fail(SPG_ERR_UNSUPPORTED, "%s: quant_rows must equal block (per-block scales), or be 32 with block = 128 and no "
                "mean (per-warp scales of Q); got quant_rows = %d, block = %d, km %s", fn, quant_rows, block,
                km == nullptr ? "NULL" : "given");
  SPG_NONNULL(fn, x); SPG_NONNULL(fn, xq); SPG_NONNULL(fn, scale);
  if ((pool == nullptr) != (sim == nullptr)) return fail(SPG_ERR_INVALID, "%s: pool and sim must both be given or both be NULL", fn);
  if (pool != nullptr) SPG_NONNULL(fn, simthreshd1);
  spg::Strides xs;
  SPG_TRY(get_strides(fn, "x_strides", x_strides, H, N, D, &xs));
  spg::launch_pool_sim_quant(x, xs, km, pool, sim, xq, scale, simthreshd1, B, H, N, D, block, quant_rows, dtype,
                             (hipStream_t)stream);
  return check_launch(fn, hipSuccess);
}

int spg_block_select(const void *pool_q, const uint8_t *sim_q, const void *pool_k, const uint8_t *sim_k,
                     const float *topk, const float *cdfthreshd, int is_causal, int attention_sink, int32_t *lut,
                     int32_t *valid_block_num, uint8_t *block_map, int B, int H, int Hkv, int nq, int nk, int D, int dtype,
                     void *stream) {
  const char *fn = "spg_block_select";
  if (B <= 0 || H <= 0 || nq <= 0 || nk <= 0) return fail(SPG_ERR_INVALID, "%s: B, H, nq, nk must be positive", fn);
  SPG_TRY(check_kv_heads(fn, H, Hkv));
  if (D != 64 && D != 128) return fail(SPG_ERR_UNSUPPORTED, "%s: head_dim must be 64 or 128 (got %d)", fn, D);
  SPG_TRY(check_dtype(fn, dtype));
  if ((topk == nullptr) == (cdfthreshd == nullptr))
    return fail(SPG_ERR_INVALID, "%s: Only one of cdfthreshd and topk can be set.", fn);
  if (nk > spg::block_select_max_nk())
    return fail(SPG_ERR_UNSUPPORTED, "%s: nk = %d exceeds the supported maximum %d", fn, nk, spg::block_select_max_nk());
  SPG_NONNULL(fn, pool_q); SPG_NONNULL(fn, sim_q); SPG_NONNULL(fn, pool_k); SPG_NONNULL(fn, sim_k);
  SPG_NONNULL(fn, lut); SPG_NONNULL(fn, valid_block_num);
  return check_launch(fn, spg::launch_block_select(pool_q, sim_q, pool_k, sim_k, topk, cdfthreshd, is_causal ? 1 : 0,
                                                   attention_sink ? 1 : 0, lut, valid_block_num, block_map, B, H, Hkv,
                                                   nq, nk, D, dtype, (hipStream_t)stream));
}

int spg_map_to_lut(const void *mask, int mask_kind, int32_t *lut, int32_t *valid_block_num, int B, int H, int nq,
                   int nk, void *stream) {
  const char *fn = "spg_map_to_lut";
  if (B <= 0 || H <= 0 || nq <= 0 || nk <= 0) return fail(SPG_ERR_INVALID, "%s: B, H, nq, nk must be positive", fn);
  if (mask_kind < SPG_MASK_I8 || mask_kind > SPG_MASK_F64) return fail(SPG_ERR_INVALID, "%s: bad mask_kind %d", fn, mask_kind);
  if (nk > 32768) return fail(SPG_ERR_UNSUPPORTED, "%s: nk = %d exceeds the supported maximum 32768", fn, nk);
  SPG_NONNULL(fn, mask); SPG_NONNULL(fn, lut); SPG_NONNULL(fn, valid_block_num);
  return check_launch(fn, spg::launch_map_to_lut(mask, mask_kind, lut, valid_block_num, B, H, nq, nk, (hipStream_t)stream));
}

int spg_selftest_division(unsigned long long *counts, int n_divisors, unsigned int seed, void *stream) {
  const char *fn = "spg_selftest_division";
  if (n_divisors <= 0 || n_divisors > (1 << 22)) return fail(SPG_ERR_INVALID, "%s: n_divisors must be in [1, 2^22]", fn);
  SPG_NONNULL(fn, counts);
  spg::launch_div_selftest(counts, n_divisors, seed, (hipStream_t)stream);
  return check_launch(fn, hipSuccess);
}

int spg_selftest_fp8_pack(const float *x, uint8_t *codes, int n, int saturate, void *stream) {
  const char *fn = "spg_selftest_fp8_pack";
  if (n <= 0 || n % 4 != 0) return fail(SPG_ERR_INVALID, "%s: n must be a positive multiple of 4 (got %d)", fn, n);
  SPG_NONNULL(fn, x); SPG_NONNULL(fn, codes);
  spg::launch_fp8_pack_selftest(x, codes, n, saturate ? 1 : 0, (hipStream_t)stream);
  return check_launch(fn, hipSuccess);
}

int spg_v_quant_fp8(const void *v, const int64_t *v_strides, uint8_t *v8, float *v_scale, int B, int H, int N, int D, int dtype, void *stream) {
  const char *fn = "spg_v_quant_fp8";
  SPG_TRY(check_shape(fn, B, H, N, D));
  SPG_TRY(check_dtype(fn, dtype));
  SPG_NONNULL(fn, v); SPG_NONNULL(fn, v8); SPG_NONNULL(fn, v_scale);
  spg::Strides vs;
  SPG_TRY(get_strides(fn, "v_strides", v_strides, H, N, D, &vs));
  spg::launch_v_quant_fp8(v, vs, v8, v_scale, B, H, N, D, dtype, (hipStream_t)stream);
  return check_launch(fn, hipSuccess);
}

int spg_block_sparse_attn(const int8_t *q8, const int8_t *k8, const uint8_t *v8, void *out, const int64_t *out_strides,
                          int out_dtype,
                          const int32_t *lut, const int32_t *valid_block_num, const float *pvthreshd,
                          const float *q_scale, const float *k_scale, const float *v_scale, int B, int H, int Hkv, int N,
                          int N_kv, int D, float sm_scale, int is_causal, int qk_quant_gran, int pv_threshold_mode,
                          int32_t *pv_count, void *stream) {
  const char *fn = "spg_block_sparse_attn";
  SPG_TRY(check_shape(fn, B, H, N, D));
  SPG_TRY(check_shape(fn, B, Hkv > 0 ? Hkv : 1, N_kv, D));
  SPG_TRY(check_kv_heads(fn, H, Hkv));
  SPG_TRY(check_quant_gran(fn, qk_quant_gran));
  SPG_TRY(check_pv_mode(fn, pv_threshold_mode));
  SPG_TRY(check_dtype(fn, out_dtype));
  SPG_NONNULL(fn, q8); SPG_NONNULL(fn, k8); SPG_NONNULL(fn, v8); SPG_NONNULL(fn, out); SPG_NONNULL(fn, lut);
  SPG_NONNULL(fn, valid_block_num); SPG_NONNULL(fn, pvthreshd); SPG_NONNULL(fn, q_scale); SPG_NONNULL(fn, k_scale);
  SPG_NONNULL(fn, v_scale);
  spg::Strides os;
  SPG_TRY(get_strides(fn, "out_strides", out_strides, H, N, D, &os));
  return check_launch(fn, spg::launch_block_sparse_attn(q8, k8, v8, out, os, out_dtype, lut, valid_block_num, pvthreshd,
                                                        q_scale, k_scale, v_scale, B, H, Hkv, N, N_kv, D, sm_scale,
                                                        is_causal ? 1 : 0, qk_quant_gran == SPG_QUANT_PER_WARP ? 1 : 0,
                                                        pv_threshold_mode, pv_count, (hipStream_t)stream));
}

int spg_v_tiles_f16(const void *v, const int64_t *v_strides, void *vt, int B, int H, int N, int D, int dtype, void *stream) {
  const char *fn = "spg_v_tiles_f16";
  SPG_TRY(check_shape(fn, B, H, N, D));
  SPG_TRY(check_dtype(fn, dtype));
  SPG_NONNULL(fn, v); SPG_NONNULL(fn, vt);
  spg::Strides vs;
  SPG_TRY(get_strides(fn, "v_strides", v_strides, H, N, D, &vs));
  spg::launch_v_tiles_f16(v, vs, vt, B, H, N, D, dtype, (hipStream_t)stream);
  return check_launch(fn, hipSuccess);
}

int spg_block_sparse_attn_f16v(const int8_t *q8, const int8_t *k8, const void *vt, void *out, const int64_t *out_strides,
                               int out_dtype,
                               const int32_t *lut, const int32_t *valid_block_num, const float *pvthreshd,
                               const float *q_scale, const float *k_scale, int B, int H, int Hkv, int N, int N_kv, int D,
                               float sm_scale, int is_causal, int qk_quant_gran, int pv_threshold_mode, int32_t *pv_count,
                               void *stream) {
  const char *fn = "spg_block_sparse_attn_f16v";
  SPG_TRY(check_shape(fn, B, H, N, D));
  SPG_TRY(check_shape(fn, B, Hkv > 0 ? Hkv : 1, N_kv, D));
  SPG_TRY(check_kv_heads(fn, H, Hkv));
  SPG_TRY(check_quant_gran(fn, qk_quant_gran));
  SPG_TRY(check_pv_mode(fn, pv_threshold_mode));
  SPG_TRY(check_dtype(fn, out_dtype));
  SPG_NONNULL(fn, q8); SPG_NONNULL(fn, k8); SPG_NONNULL(fn, vt); SPG_NONNULL(fn, out); SPG_NONNULL(fn, lut);
  SPG_NONNULL(fn, valid_block_num); SPG_NONNULL(fn, pvthreshd); SPG_NONNULL(fn, q_scale); SPG_NONNULL(fn, k_scale);
  spg::Strides os;
  SPG_TRY(get_strides(fn, "out_strides", out_strides, H, N, D, &os));
  return check_launch(fn, spg::launch_block_sparse_attn(q8, k8, (const uint8_t *)vt, out, os, out_dtype, lut, valid_block_num,
                                                        pvthreshd, q_scale, k_scale, nullptr, B, H, Hkv, N, N_kv, D, sm_scale,
                                                        is_causal ? 1 : 0, qk_quant_gran == SPG_QUANT_PER_WARP ? 1 : 0,
                                                        pv_threshold_mode, pv_count, (hipStream_t)stream));
}

int spg_few_rows_route(int B, int H, int N, int N_kv, int D, int pv_f16, int selection, float share, float simthreshd1, int is_causal,
                       float pvthreshd, uint64_t *workspace_bytes) {
  const char *fn = "spg_few_rows_route";
  if (workspace_bytes != nullptr) *workspace_bytes = 0;
  if (check_shape(fn, B, H, N, D) != SPG_OK || check_shape(fn, B, H, N_kv, D) != SPG_OK) return SPG_ROWS_ONE_WORKGROUP;
  if (few_rows(B, H, N, N_kv, D, pv_f16 != 0, pvthreshd) > 0) return SPG_ROWS_BY_QUERIES;
  if (!rows_in_chunks(B, H, N, N_kv, D, pv_f16 != 0, selection, share, simthreshd1, is_causal != 0)) return SPG_ROWS_ONE_WORKGROUP;
  if (workspace_bytes != nullptr) *workspace_bytes = chunk_plan(B, H, N, N_kv, D).bytes;
  return SPG_ROWS_BY_BLOCKS;
}

int spg_block_sparse_attn_few_rows(const int8_t *q8, const int8_t *k8, const void *v, void *out, const int64_t *out_strides, int out_dtype,
                                   const int32_t *lut, const int32_t *valid_block_num, const float *pvthreshd, const float *q_scale,
                                   const float *k_scale, const float *v_scale, int B, int H, int Hkv, int N, int N_kv, int D, float sm_scale,
                                   int is_causal, int qk_quant_gran, int route, void *workspace, uint64_t workspace_bytes, void *stream) {
  const char *fn = "spg_block_sparse_attn_few_rows";
  SPG_TRY(check_shape(fn, B, H, N, D));
  SPG_TRY(check_shape(fn, B, Hkv > 0 ? Hkv : 1, N_kv, D));
  SPG_TRY(check_kv_heads(fn, H, Hkv));
  SPG_TRY(check_quant_gran(fn, qk_quant_gran));
  SPG_TRY(check_dtype(fn, out_dtype));
  SPG_NONNULL(fn, q8); SPG_NONNULL(fn, k8); SPG_NONNULL(fn, v); SPG_NONNULL(fn, out); SPG_NONNULL(fn, lut);
  SPG_NONNULL(fn, valid_block_num); SPG_NONNULL(fn, pvthreshd); SPG_NONNULL(fn, q_scale); SPG_NONNULL(fn, k_scale);
  spg::Strides os;
  SPG_TRY(get_strides(fn, "out_strides", out_strides, H, N, D, &os));
  const ChunkPlan c = chunk_plan(B, H, N, N_kv, D);
  const int few = few_rows(B, H, N, N_kv, D, v_scale == nullptr, INFINITY);
  if (route != SPG_ROWS_BY_QUERIES && route != SPG_ROWS_BY_BLOCKS) return fail(SPG_ERR_INVALID, "%s: bad route %d", fn, route);
  if (route == SPG_ROWS_BY_QUERIES ? few == 0 : c.chunks == 1) return fail(SPG_ERR_UNSUPPORTED, "%s: the rows of this call have one workgroup each", fn);
  RowSplit split = {};
  if (route == SPG_ROWS_BY_BLOCKS) {
    SPG_NONNULL(fn, workspace);
    if (workspace_bytes < c.bytes) return fail(SPG_ERR_INVALID, "%s: workspace of %zu bytes, %zu needed", fn, (size_t)workspace_bytes, c.bytes);
    if ((uintptr_t)workspace % 256 != 0) return fail(SPG_ERR_INVALID, "%s: workspace must be 256-byte aligned (got %p)", fn, workspace);
    split = row_split(c, workspace);
  }
  return check_launch(fn, spg::launch_block_sparse_attn_h(q8, k8, (const uint8_t *)v, out, os, out_dtype, lut, valid_block_num, nullptr, nullptr,
                                                          Hyper{pvthreshd, 0.f}, q_scale, k_scale, v_scale, B, H, Hkv, N, N_kv, D, sm_scale,
                                                          is_causal ? 1 : 0, qk_quant_gran == SPG_QUANT_PER_WARP ? 1 : 0, SPG_PV_PER_BLOCK,
                                                          nullptr, false, nullptr, &split, route == SPG_ROWS_BY_QUERIES ? few : 0, (hipStream_t)stream));
}

static int check_forward(const char *fn, const spg_attn_args *a) {
  SPG_TRY(check_shape(fn, a->B, a->H, a->N, a->D));
  SPG_TRY(check_shape(fn, a->B, a->Hkv > 0 ? a->Hkv : 1, a->N_kv, a->D));
  SPG_TRY(check_kv_heads(fn, a->H, a->Hkv));
  SPG_TRY(check_dtype(fn, a->qk_dtype));
  SPG_TRY(check_dtype(fn, a->v_dtype));
  SPG_TRY(check_quant_gran(fn, a->qk_quant_gran));
  if (a->selection < SPG_SELECT_TOPK || a->selection > SPG_SELECT_MASK)
    return fail(SPG_ERR_INVALID, "%s: selection must be 0 (top-k), 1 (CDF) or 2 (mask), got %d", fn, a->selection);
  const int nk = (a->N_kv + 63) / 64;
  if (a->selection == SPG_SELECT_MASK) {
    if (a->mask_kind < SPG_MASK_I8 || a->mask_kind > SPG_MASK_F64) return fail(SPG_ERR_INVALID, "%s: bad mask_kind %d", fn, a->mask_kind);
    if (nk > 32768) return fail(SPG_ERR_UNSUPPORTED, "%s: nk = %d exceeds the supported maximum 32768", fn, nk);
  } else if (nk > spg::block_select_max_nk()) {
    return fail(SPG_ERR_UNSUPPORTED, "%s: nk = %d exceeds the supported maximum %d", fn, nk, spg::block_select_max_nk());
  }
  return SPG_OK;
}

// The counts of a call on its own are there after 20 to 40 us, behind an earlier call of the same kind after 100 to 200: they are looked
// for without a pause.  After half a millisecond the call stands behind other work (or the memory is not coherent, and the counts come
// with the end of the kernel): the core is given back, and looking every 50 us adds little to a wait of that length.
int64_t spg_wait_counts(const int32_t *counts, int64_t n, double seconds) {
  if (counts == nullptr || n < 0) return -1;
  const auto start = std::chrono::steady_clock::now();
  int64_t sum = 0, i = 0;
  for (unsigned spin = 1;; spin++) {
    for (int v; i < n && (v = __atomic_load_n(counts + i, __ATOMIC_ACQUIRE)) >= 0; i++) sum += v;
    if (i == n) return sum;
    if (spin % 64 != 0) continue;
    const double waited = std::chrono::duration<double>(std::chrono::steady_clock::now() - start).count();
    if (waited > seconds) return -1;
    if (waited > 5e-4) {
      std::this_thread::sleep_for(std::chrono::microseconds(50));
      spin = 63;                                     // look once, then at the clock again
    }
  }
}

size_t spg_sparse_attn_workspace_bytes(const spg_attn_args *args) {
  if (args == nullptr || check_forward("spg_sparse_attn_workspace_bytes", args) != SPG_OK) return 0;
  return layout_for(args).total;
}

int spg_sparse_attn(const spg_attn_args *args, void *stream) {
  const char *fn = "spg_sparse_attn";
  SPG_NONNULL(fn, args);
  const spg_attn_args *a = args;
  SPG_TRY(check_forward(fn, a));
  SPG_NONNULL(fn, a->q); SPG_NONNULL(fn, a->k); SPG_NONNULL(fn, a->v); SPG_NONNULL(fn, a->out); SPG_NONNULL(fn, a->workspace);
  if (a->selection == SPG_SELECT_MASK) SPG_NONNULL(fn, a->mask);
  const size_t need = layout_for(a).total;
  if (a->workspace_bytes < need) return fail(SPG_ERR_INVALID, "%s: workspace of %zu bytes, %zu needed", fn, (size_t)a->workspace_bytes, need);
  // every part of the workspace starts at a multiple of 256 bytes and is read and written in pieces of up to 16
  if ((uintptr_t)a->workspace % 256 != 0) return fail(SPG_ERR_INVALID, "%s: workspace must be 256-byte aligned (got %p)", fn, a->workspace);
  Strides qs, ks, vs, os;
  SPG_TRY(get_strides(fn, "q_strides", a->q_strides, a->H, a->N, a->D, &qs));
  SPG_TRY(get_strides(fn, "k_strides", a->k_strides, a->Hkv, a->N_kv, a->D, &ks));
  SPG_TRY(get_strides(fn, "v_strides", a->v_strides, a->Hkv, a->N_kv, a->D, &vs));
  SPG_TRY(get_strides(fn, "out_strides", a->out_strides, a->H, a->N, a->D, &os));
  return check_launch(fn, run_forward(a, qs, ks, vs, os, (hipStream_t)stream));
}

int spg_dense_attn_f16(const void *q, const void *k, const void *v, void *out, int B, int H, int N, int D,
                       float sm_scale, int is_causal, void *stream) {
  const char *fn = "spg_dense_attn_f16";
  SPG_TRY(check_shape(fn, B, H, N, D));
  SPG_NONNULL(fn, q); SPG_NONNULL(fn, k); SPG_NONNULL(fn, v); SPG_NONNULL(fn, out);
  return check_launch(fn, spg::launch_dense_attn_f16(q, k, v, out, B, H, N, D, sm_scale, is_causal ? 1 : 0,
                                                     (hipStream_t)stream));
}

}  // extern "C"
