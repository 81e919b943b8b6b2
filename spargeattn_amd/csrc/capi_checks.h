// Argument checks shared by the extern "C" entry points (capi.hip, forward.hip).
#pragma once
#include "../../include/spargeattn_amd.h"
#include "launch.h"

namespace spg {

// writes the calling thread's error message (spg_last_error) and returns `code`
int fail(int code, const char *fmt, ...) __attribute__((visibility("hidden")));

inline int check_launch(const char *what, hipError_t e) {
  if (e == hipSuccess) e = hipGetLastError();
  if (e != hipSuccess) return fail(SPG_ERR_HIP, "%s: %s", what, hipGetErrorString(e));
  return SPG_OK;
}

inline int check_shape(const char *fn, int B, int H, int N, int D) {
  if (B <= 0 || H <= 0 || N <= 0) return fail(SPG_ERR_INVALID, "%s: B, H, N must be positive (got %d, %d, %d)", fn, B, H, N);
  if (D != 64 && D != 128) return fail(SPG_ERR_UNSUPPORTED, "%s: head_dim must be 64 or 128 (got %d)", fn, D);
  if ((double)B * H * (double)N * D >= 4294967296.0 * 4)
    return fail(SPG_ERR_UNSUPPORTED, "%s: tensor too large (B*H*N*D = %.0f)", fn, (double)B * H * (double)N * D);
  return SPG_OK;
}

inline int check_kv_heads(const char *fn, int H, int Hkv) {
  // the message of the reference (qk_int_sv_f8_cuda_sm89.cu:310-314)
  if (Hkv <= 0 || H % Hkv != 0)
    return fail(SPG_ERR_INVALID, "%s: num_qo_heads (%d) must be divisible by num_kv_heads (%d)", fn, H, Hkv);
  return SPG_OK;
}

inline int check_pv_mode(const char *fn, int mode) {
  if (mode < SPG_PV_NONE || mode > SPG_PV_PER_WARP)
    return fail(SPG_ERR_INVALID, "%s: pv_threshold_mode must be 0 (none), 1 (per block) or 2 (per 32 query rows), got %d", fn, mode);
  return SPG_OK;
}

// qk_quant_gran of the reference's kernel entry (csrc/pytorch_extensions_utils.cuh:71-85): 1 per block, 2 per warp,
// 3 per thread.  Per-thread scales follow the lane layout of mma.sync fragments and have no counterpart here.
inline int check_quant_gran(const char *fn, int gran) {
  if (gran == SPG_QUANT_PER_BLOCK || gran == SPG_QUANT_PER_WARP) return SPG_OK;
  if (gran == 3) return fail(SPG_ERR_UNSUPPORTED, "%s: qk_quant_gran 3 (per thread) is not supported on gfx950", fn);
  return fail(SPG_ERR_INVALID, "%s: Unsupported qk_quant_gran: %d", fn, gran);
}

inline int check_dtype(const char *fn, int dtype) {
  if (dtype != SPG_F16 && dtype != SPG_BF16) return fail(SPG_ERR_INVALID, "%s: dtype must be SPG_F16 or SPG_BF16 (got %d)", fn, dtype);
  return SPG_OK;
}

// strides == NULL: HND-contiguous.  Otherwise {batch, head, row} strides in elements; rows are read and written in
// 16-byte pieces, so every stride must be a multiple of 8 elements and a row must not overlap the next one.
inline int get_strides(const char *fn, const char *what, const int64_t *strides, int H, int N, int D, Strides *out) {
  if (strides == nullptr) {
    out->sb = (long long)H * N * D; out->sh = (long long)N * D; out->sn = D;
    return SPG_OK;
  }
  for (int i = 0; i < 3; i++)
    if (strides[i] <= 0 || strides[i] % 8 != 0)
      return fail(SPG_ERR_INVALID, "%s: %s[%d] = %lld must be a positive multiple of 8 elements", fn, what, i, (long long)strides[i]);
  if (strides[2] < D) return fail(SPG_ERR_INVALID, "%s: %s[2] = %lld is smaller than head_dim %d", fn, what, (long long)strides[2], D);
  out->sb = strides[0]; out->sh = strides[1]; out->sn = strides[2];
  return SPG_OK;
}

#define SPG_TRY(expr) do { int rc_ = (expr); if (rc_ != SPG_OK) return rc_; } while (0)
#define SPG_NONNULL(fn, ptr) do { if ((ptr) == nullptr) return fail(SPG_ERR_INVALID, "%s: %s is NULL", fn, #ptr); } while (0)

}  // namespace spg
