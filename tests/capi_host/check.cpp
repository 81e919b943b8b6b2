// Runs the host-side argument validation of the C ABI (spargeattn_amd/csrc/capi.hip) with bad arguments of every kind.
// Built with -fsanitize=address,undefined by tests/test_capi_sanitized.py: a validation path that reads a stride array
// out of bounds, formats a message past its buffer or overflows a size computation fails the run.  No GPU is touched:
// every call must be refused before a launch (spg::g_launches stays 0), but for the one that says so.
#include "../../include/spargeattn_amd.h"

#include <cstdio>
#include <cstring>

namespace spg { extern int g_launches; }

static int failures = 0;
#define EXPECT(rc, code, needle)                                                                         \
  do {                                                                                                   \
    const int rc_ = (rc);                                                                                \
    if (rc_ != (code) || std::strstr(spg_last_error(), (needle)) == nullptr) {                           \
      std::printf("line %d: rc %d (want %d), message '%s' (want '%s')\n", __LINE__, rc_, (int)(code), spg_last_error(), (needle)); \
      failures++;                                                                                        \
    }                                                                                                    \
  } while (0)

int main() {
  void *p = (void *)0x1000;                 // never dereferenced: every call below is refused on its arguments
  const float *fp = (const float *)p;
  int8_t *i8 = (int8_t *)p;
  uint8_t *u8 = (uint8_t *)p;
  int32_t *i32 = (int32_t *)p;
  int64_t bad_mult[3] = {128 * 64, 64, 60}, bad_small[3] = {128 * 64, 128 * 64, 32}, neg[3] = {-8, 64, 64};
  int64_t huge[3] = {INT64_MAX - 7, 8, 64};

  EXPECT(spg_km_mean(nullptr, nullptr, nullptr, nullptr, 1, 1, 128, 96, 0, nullptr), SPG_ERR_UNSUPPORTED, "head_dim");
  EXPECT(spg_km_mean(p, nullptr, p, p, 0, 1, 128, 64, 0, nullptr), SPG_ERR_INVALID, "must be positive");
  EXPECT(spg_km_mean(p, nullptr, p, p, 65536, 65536, 1 << 30, 128, 0, nullptr), SPG_ERR_UNSUPPORTED, "too large");
  EXPECT(spg_km_mean(p, nullptr, p, nullptr, 1, 1, 128, 64, 0, nullptr), SPG_ERR_INVALID, "NULL");
  EXPECT(spg_km_mean(p, bad_mult, p, p, 1, 1, 128, 64, 0, nullptr), SPG_ERR_INVALID, "multiple of 8");
  EXPECT(spg_km_mean(p, bad_small, p, p, 1, 1, 128, 64, 0, nullptr), SPG_ERR_INVALID, "smaller than head_dim");
  EXPECT(spg_km_mean(p, neg, p, p, 1, 1, 128, 64, 0, nullptr), SPG_ERR_INVALID, "positive multiple");
  EXPECT(spg_km_mean(p, huge, p, p, 1, 1, 128, 64, 7, nullptr), SPG_ERR_INVALID, "dtype");
  EXPECT(spg_km_mean_static(p, nullptr, p, 1, 8193, 128, 128, 0, nullptr), SPG_ERR_UNSUPPORTED, "scratch");
  if (spg_km_mean_workspace_bytes(-1, 1, 1, 1) != 0 || spg_km_mean_workspace_bytes(1, 32, 32768, 128) == 0) failures++;

  EXPECT(spg_pool_sim_quant(nullptr, nullptr, nullptr, nullptr, nullptr, nullptr, nullptr, nullptr, 1, 1, 128, 64, 128, 128, 1, nullptr),
         SPG_ERR_INVALID, "NULL");
  EXPECT(spg_pool_sim_quant(p, nullptr, nullptr, p, nullptr, i8, (float *)p, fp, 1, 1, 128, 64, 128, 128, 1, nullptr),
         SPG_ERR_INVALID, "both be given");
  EXPECT(spg_pool_sim_quant(p, nullptr, nullptr, nullptr, nullptr, i8, (float *)p, nullptr, 1, 1, 128, 64, 96, 96, 1, nullptr),
         SPG_ERR_UNSUPPORTED, "block must be");
  EXPECT(spg_pool_sim_quant(p, nullptr, nullptr, nullptr, nullptr, i8, (float *)p, nullptr, 1, 1, 128, 64, 64, 32, 1, nullptr),
         SPG_ERR_UNSUPPORTED, "quant_rows");
  EXPECT(spg_pool_sim_quant(p, nullptr, p, nullptr, nullptr, i8, (float *)p, nullptr, 1, 1, 128, 64, 128, 32, 1, nullptr),
         SPG_ERR_UNSUPPORTED, "quant_rows");

  EXPECT(spg_block_select(p, u8, p, u8, nullptr, nullptr, 0, 0, i32, i32, nullptr, 1, 1, 1, 1, 2, 64, 0, nullptr), SPG_ERR_INVALID,
         "Only one of cdfthreshd and topk");
  EXPECT(spg_block_select(p, u8, p, u8, fp, fp, 0, 0, i32, i32, nullptr, 1, 1, 1, 1, 2, 64, 0, nullptr), SPG_ERR_INVALID,
         "Only one of cdfthreshd and topk");
  EXPECT(spg_block_select(p, u8, p, u8, fp, nullptr, 0, 0, i32, i32, nullptr, 1, 6, 4, 1, 2, 64, 0, nullptr), SPG_ERR_INVALID,
         "must be divisible by num_kv_heads");
  EXPECT(spg_block_select(p, u8, p, u8, fp, nullptr, 0, 0, i32, i32, nullptr, 1, 6, 0, 1, 2, 64, 0, nullptr), SPG_ERR_INVALID,
         "must be divisible by num_kv_heads");
  EXPECT(spg_block_select(p, u8, p, u8, fp, nullptr, 0, 0, i32, i32, nullptr, 1, 4, 4, 1, 8193, 64, 0, nullptr), SPG_ERR_UNSUPPORTED,
         "exceeds the supported maximum");
  EXPECT(spg_map_to_lut(p, 9, i32, i32, 1, 1, 1, 1, nullptr), SPG_ERR_INVALID, "bad mask_kind");
  EXPECT(spg_map_to_lut(p, 0, i32, i32, 1, 1, 1, 40000, nullptr), SPG_ERR_UNSUPPORTED, "exceeds the supported maximum");

  EXPECT(spg_v_quant_fp8(p, nullptr, u8, (float *)p, 1, 1, 128, 64, 7, nullptr), SPG_ERR_INVALID, "dtype");
  EXPECT(spg_v_quant_fp8(p, bad_mult, u8, (float *)p, 1, 1, 128, 64, 0, nullptr), SPG_ERR_INVALID, "multiple of 8");
  EXPECT(spg_v_tiles_f16(p, bad_small, p, 1, 1, 128, 64, 0, nullptr), SPG_ERR_INVALID, "smaller than head_dim");

  for (int f16v = 0; f16v < 2; f16v++) {
    auto attn = [&](int H, int Hkv, int N, int Nkv, int D, int gran, int pv) {
      return f16v ? spg_block_sparse_attn_f16v(i8, i8, p, p, nullptr, 0, i32, i32, fp, fp, fp, 1, H, Hkv, N, Nkv, D, 0.125f, 0,
                                                gran, pv, nullptr, nullptr)
                  : spg_block_sparse_attn(i8, i8, u8, p, nullptr, 0, i32, i32, fp, fp, fp, fp, 1, H, Hkv, N, Nkv, D, 0.125f, 0, gran,
                                          pv, nullptr, nullptr);
    };
    EXPECT(attn(6, 4, 128, 128, 64, 1, 1), SPG_ERR_INVALID, "must be divisible by num_kv_heads");
    EXPECT(attn(4, 4, 128, 128, 64, 1, 3), SPG_ERR_INVALID, "pv_threshold_mode");
    EXPECT(attn(4, 4, 128, 0, 64, 1, 1), SPG_ERR_INVALID, "must be positive");
    EXPECT(attn(4, 4, 128, 128, 80, 1, 1), SPG_ERR_UNSUPPORTED, "head_dim");
    EXPECT(attn(4, 4, 128, 128, 64, 3, 1), SPG_ERR_UNSUPPORTED, "per thread");
    EXPECT(attn(4, 4, 128, 128, 64, 0, 1), SPG_ERR_INVALID, "Unsupported qk_quant_gran: 0");
    EXPECT(attn(4, 4, 128, 128, 64, -7, 1), SPG_ERR_INVALID, "Unsupported qk_quant_gran: -7");
  }
  EXPECT(spg_block_sparse_attn(i8, i8, u8, p, neg, 0, i32, i32, fp, fp, fp, fp, 1, 4, 4, 128, 128, 64, 0.125f, 0, 1, 1, nullptr, nullptr),
         SPG_ERR_INVALID, "positive multiple");
  EXPECT(spg_dense_attn_f16(p, p, nullptr, p, 1, 1, 128, 64, 0.125f, 0, nullptr), SPG_ERR_INVALID, "NULL");
  EXPECT(spg_selftest_fp8_pack(fp, u8, 6, 1, nullptr), SPG_ERR_INVALID, "multiple of 4");
  EXPECT(spg_selftest_division(nullptr, 16, 1, nullptr), SPG_ERR_INVALID, "NULL");
  EXPECT(spg_selftest_division((unsigned long long *)p, 0, 1, nullptr), SPG_ERR_INVALID, "n_divisors");

  // the whole operator: every field of its argument block that is checked, one at a time against a block that is accepted
  spg_attn_args good = {};
  good.B = 2; good.H = 4; good.Hkv = 2; good.N = 300; good.N_kv = 700; good.D = 64;
  good.qk_dtype = SPG_F16; good.v_dtype = SPG_BF16; good.selection = SPG_SELECT_TOPK; good.qk_quant_gran = SPG_QUANT_PER_BLOCK;
  good.q = good.k = good.v = good.mask = p; good.out = p; good.workspace = p;
  good.workspace_bytes = spg_sparse_attn_workspace_bytes(&good);
  if (good.workspace_bytes == 0) failures++;
  EXPECT(spg_sparse_attn(nullptr, nullptr), SPG_ERR_INVALID, "NULL");
  if (spg_sparse_attn_workspace_bytes(nullptr) != 0) failures++;
  // sizes and options: both entry points refuse them
#define REFUSED(change, code, needle)                                                                    \
  {                                                                                                      \
    spg_attn_args a = good;                                                                              \
    change;                                                                                              \
    EXPECT(spg_sparse_attn(&a, nullptr), code, needle);                                                  \
    if (spg_sparse_attn_workspace_bytes(&a) != 0) { std::printf("line %d: a workspace size for " #change "\n", __LINE__); failures++; } \
  }
  REFUSED(a.B = 0, SPG_ERR_INVALID, "must be positive")
  REFUSED(a.N = -5, SPG_ERR_INVALID, "must be positive")
  REFUSED(a.N_kv = 0, SPG_ERR_INVALID, "must be positive")
  REFUSED(a.D = 96, SPG_ERR_UNSUPPORTED, "head_dim")
  REFUSED(a.N = INT32_MAX, SPG_ERR_UNSUPPORTED, "too large")
  REFUSED(a.N_kv = INT32_MAX, SPG_ERR_UNSUPPORTED, "too large")
  REFUSED(a.Hkv = 3, SPG_ERR_INVALID, "must be divisible by num_kv_heads")
  REFUSED(a.Hkv = 0, SPG_ERR_INVALID, "must be divisible by num_kv_heads")
  REFUSED(a.Hkv = -2, SPG_ERR_INVALID, "must be divisible by num_kv_heads")
  REFUSED(a.qk_dtype = 2, SPG_ERR_INVALID, "dtype")
  REFUSED(a.v_dtype = -1, SPG_ERR_INVALID, "dtype")
  REFUSED(a.qk_quant_gran = 0, SPG_ERR_INVALID, "Unsupported qk_quant_gran: 0")
  REFUSED(a.qk_quant_gran = 3, SPG_ERR_UNSUPPORTED, "per thread")
  REFUSED(a.selection = 3, SPG_ERR_INVALID, "selection")
  REFUSED(a.selection = -1, SPG_ERR_INVALID, "selection")
  REFUSED((a.selection = SPG_SELECT_MASK, a.mask_kind = 7), SPG_ERR_INVALID, "bad mask_kind")
  REFUSED((a.selection = SPG_SELECT_MASK, a.N_kv = 32769 * 64), SPG_ERR_UNSUPPORTED, "exceeds the supported maximum 32768")
  REFUSED(a.N_kv = 8193 * 64, SPG_ERR_UNSUPPORTED, "exceeds the supported maximum 8192")
#undef REFUSED
  // pointers, workspace and strides: the call refuses them
#define REFUSED(change, needle)                                                                          \
  {                                                                                                      \
    spg_attn_args a = good;                                                                              \
    change;                                                                                              \
    EXPECT(spg_sparse_attn(&a, nullptr), SPG_ERR_INVALID, needle);                                       \
  }
  REFUSED(a.q = nullptr, "a->q is NULL")
  REFUSED(a.k = nullptr, "a->k is NULL")
  REFUSED(a.v = nullptr, "a->v is NULL")
  REFUSED(a.out = nullptr, "a->out is NULL")
  REFUSED(a.workspace = nullptr, "a->workspace is NULL")
  REFUSED((a.selection = SPG_SELECT_MASK, a.mask = nullptr), "a->mask is NULL")
  REFUSED((a.workspace = (char *)p + 128, a.workspace_bytes += 128), "256-byte aligned")
  REFUSED(a.workspace_bytes -= 1, "needed")
  REFUSED((a.pv_f16 = 1), "needed")                       // FP16 tiles take more than the workspace of the FP8 form
  REFUSED(a.q_strides = bad_mult, "q_strides[2]")
  REFUSED(a.k_strides = neg, "k_strides[0]")
  REFUSED(a.v_strides = bad_small, "v_strides[2]")
  REFUSED(a.out_strides = bad_mult, "out_strides[2]")
#undef REFUSED
  if (spg::g_launches != 0) { std::printf("a refused call reached a launcher (%d)\n", spg::g_launches); failures++; }
  // workspace sizes at the ends of what is accepted: no overflow, room for the int8 tensors, more for more work
  {
    const struct { int B, H, Hkv, N, N_kv, D; } shapes[] = {{1, 1, 1, 1, 1, 64}, {1, 1, 1, 128, 64 * 8192, 128}, {1, 1, 1, 1 << 27, 64, 64},
                                                            {1 << 14, 1 << 13, 1, 1, 1, 64}, {1, 1 << 27, 1 << 27, 1, 1, 64}, {1, 30, 30, 17776, 17776, 64}};
    for (const auto &s : shapes) {
      spg_attn_args a = good;
      a.B = s.B; a.H = s.H; a.Hkv = s.Hkv; a.N = s.N; a.N_kv = s.N_kv; a.D = s.D;
      const size_t n = spg_sparse_attn_workspace_bytes(&a), int8 = (size_t)s.B * s.D * ((size_t)s.H * s.N + (size_t)s.Hkv * s.N_kv);
      a.pv_f16 = 1;
      if (n < int8 || spg_sparse_attn_workspace_bytes(&a) < int8) { std::printf("workspace of %zu bytes at N %d N_kv %d\n", n, s.N, s.N_kv); failures++; }
    }
  }
  // (its status is that of the HIP runtime, which may have no device here)
  (void)spg_sparse_attn(&good, nullptr);
  if (spg::g_launches != 1) { std::printf("the accepted call was not launched once\n"); failures++; }
  spg::g_launches = 0;

  if (spg::g_launches != 0) { std::printf("a refused call reached a launcher (%d)\n", spg::g_launches); failures++; }
  if (spg_version() < 100) failures++;
  std::printf(failures ? "FAILED (%d)\n" : "capi host checks ok\n", failures);
  return failures ? 1 : 0;
}
