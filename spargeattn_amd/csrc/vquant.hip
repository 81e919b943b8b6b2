// V path for gfx950: fp16 cast, per-(b,h,channel) absmax, FP8 e4m3 quantisation written straight into the
// [B][H][nk][D][64] tile layout the attention kernel's V^T operand reads.  Inside a 64-byte tile row (one channel,
// 64 keys) the four 16-key chunks are stored XOR-swizzled: key chunk kc sits at slot kc ^ ((d >> 2) & 3), which is
// the LDS bank-conflict swizzle of the attention kernel baked into the HBM layout (a tile is copied to LDS verbatim).
// Replaces TransposePadPermuteKernel + MeanScaleKernel (csrc/fused/fused.cu:26-77, 80-191) called with
// scale_max = 2.25 (spas_sage_attn/core.py:147-151).  HBM-bound: V is read twice (absmax, quantise), written once
// at 1 B/element.  Compile with -ffp-contract=off.
#include "stage_bodies.h"

namespace spg {

__global__ void fill_u32_kernel(uint32_t *p, uint32_t v, int n) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = v;
}

template <int D, int DT>
__global__ __launch_bounds__(256) void v_absmax_kernel(const uint16_t *__restrict__ v, const Strides vs, int H,
                                                       uint32_t *__restrict__ amax_bits, int N, int rows_per_chunk) {
  __shared__ __align__(16) unsigned char smem[v_absmax_lds<D>()];
  const int bh = blockIdx.y;
  v_absmax_body<D, DT>(v, vs, H, N, rows_per_chunk, blockIdx.x, bh, smem, [&](int d, float s) {
    // non-negative floats order like their bit patterns; max is order independent
    atomicMax(amax_bits + (size_t)bh * D + d, __builtin_bit_cast(uint32_t, s));
  });
}

// One workgroup per 64-key tile.
template <int D, int DT>
__global__ __launch_bounds__(256) void v_quant_kernel(const uint16_t *__restrict__ v, const Strides vs, int H,
                                                      const float *__restrict__ amax, uint8_t *__restrict__ v8, int N, int nk) {
  __shared__ __align__(16) unsigned char smem[v_quant_lds<D>()];
  const int bh = blockIdx.y;
  v_quant_body<D, DT>(v, vs, H, v8, N, nk, blockIdx.x, bh, smem, [&](int d) { return amax[(size_t)bh * D + d]; });
}

template <int D, int DT>
__global__ __launch_bounds__(256) void v_tiles_f16_kernel(const uint16_t *__restrict__ v, const Strides vs, int H,
                                                          uint16_t *__restrict__ vt, int N, int nk) {
  __shared__ __align__(16) unsigned char smem[v_tiles_f16_lds<D>()];
  v_tiles_f16_body<D, DT>(v, vs, H, vt, N, nk, blockIdx.x, blockIdx.y, smem);
}

__global__ void v_scale_final_kernel(float *v_scale, int n) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) v_scale[i] = v_scale[i] / 2.25f;
}

static int v_chunks(int B, int H, int N) {
  int want = (4096 + B * H - 1) / (B * H);
  int maxc = (N + 255) / 256;
  int c = want < maxc ? want : maxc;
  return c < 1 ? 1 : c;
}

template <int D, int DT>
static void launch_vq2(const void *v, Strides vs, uint8_t *v8, float *v_scale, int B, int H, int N, hipStream_t st) {
  const int n = B * H * D;
  const int nk = (N + 63) / 64;
  const int nchunk = v_chunks(B, H, N);
  const int rpc = (N + nchunk - 1) / nchunk;
  fill_u32_kernel<<<(n + 255) / 256, 256, 0, st>>>((uint32_t *)v_scale, 0u, n);
  v_absmax_kernel<D, DT><<<dim3(nchunk, B * H), 256, 0, st>>>((const uint16_t *)v, vs, H, (uint32_t *)v_scale, N, rpc);
  v_quant_kernel<D, DT><<<dim3(nk, B * H), 256, 0, st>>>((const uint16_t *)v, vs, H, v_scale, v8, N, nk);
  v_scale_final_kernel<<<(n + 255) / 256, 256, 0, st>>>(v_scale, n);
}

void launch_v_quant_fp8(const void *v, Strides vs, uint8_t *v8, float *v_scale, int B, int H, int N, int D, int dtype,
                        hipStream_t st) {
  if (D == 64) { if (dtype == 0) launch_vq2<64, 0>(v, vs, v8, v_scale, B, H, N, st); else launch_vq2<64, 1>(v, vs, v8, v_scale, B, H, N, st); }
  else         { if (dtype == 0) launch_vq2<128, 0>(v, vs, v8, v_scale, B, H, N, st); else launch_vq2<128, 1>(v, vs, v8, v_scale, B, H, N, st); }
}

void launch_v_tiles_f16(const void *v, Strides vs, void *vt, int B, int H, int N, int D, int dtype, hipStream_t st) {
  const int nk = (N + 63) / 64;
  const dim3 grid(nk, B * H);
  const uint16_t *vp = (const uint16_t *)v;
  uint16_t *op = (uint16_t *)vt;
  if (D == 64) { if (dtype == 0) v_tiles_f16_kernel<64, 0><<<grid, 256, 0, st>>>(vp, vs, H, op, N, nk); else v_tiles_f16_kernel<64, 1><<<grid, 256, 0, st>>>(vp, vs, H, op, N, nk); }
  else         { if (dtype == 0) v_tiles_f16_kernel<128, 0><<<grid, 256, 0, st>>>(vp, vs, H, op, N, nk); else v_tiles_f16_kernel<128, 1><<<grid, 256, 0, st>>>(vp, vs, H, op, N, nk); }
}

}  // namespace spg
