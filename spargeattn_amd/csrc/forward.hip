// The whole operator behind one call: K mean, mask prediction + INT8 quantisation, V quantisation, block-sparse
// attention, as two to seven launches on workspace the caller hands over.
//
// Short sequences are bound by the length of the launch chain and by kernels that cannot fill the chip, so stages that do
// not depend on each other share a launch; which stage a workgroup belongs to follows from its number:
//   short    (short heads) everything up to the selection: blocks of K and V, whose workgroups sum and search their whole head for
//            themselves | mask rows | pooling + quantisation of Q.  Otherwise:
//   front    partial column sums of K | partial channel maxima of V (FP16 PV, few blocks: the V^T tiles, finished) | LUT rows of a
//            user mask | pooling + quantisation of Q (unless the attention kernel does that in place: q_in_front)
//   (final   column mean of K, channel maxima of V: only where there are too many partial results for every workgroup
//            of the next launch to add them up for itself)
//   back     pooling + quantisation of K | V -> e4m3 tiles and scales (FP16 PV, many blocks: V^T tiles)
//   select   block_select_* of maskpred.hip (rows of more than 128 blocks; shorter ones are selected inside the next launch)
//   attn     block_sparse_attn_kernel (few short rows: few_rows_attn_kernel, several workgroups to a row; few long rows: in chunks,
//            with a launch in front for their maxima and one behind)
// Every body is the one the stage-by-stage entry points launch (stage_bodies.h): results are the same bits.
// The extern "C" entry points and their argument checks are in capi.hip, the workspace layout in forward_plan.h.
// Compile with -ffp-contract=off.
#include "forward_plan.h"
#include "stage_bodies.h"

namespace spg {

constexpr int MASK_NKP_FRONT = 4096;    // longest mask row (padded to a power of two) whose index list fits the front LDS

struct FrontParams {
  const uint16_t *q, *k, *v;
  Strides qs, ks, vs;
  int H, Hkv, N, Nk, nq, nk;
  int v_dtype, v_f16;
  // first workgroup of each role; the roles follow one another in this order
  int wg_v, wg_mask, wg_q;
  int k_chunks, k_rows, v_chunks, v_rows;
  double *km_part;
  float *v_part;                        // [B Hkv][v_chunks][D]
  uint16_t *v_tiles;
  const void *mask;
  int mask_kind, nkp;
  int32_t *lut, *valid;
  Hyper simthr;
  uint16_t *pool_q;
  uint8_t *sim_q;
  int8_t *q8;
  float *q_scale;
  int *queue;                           // cleared here for the attention kernel
};

template <int A, int B> constexpr int max_c() { return A > B ? A : B; }
template <int D, bool POOL, int NT> constexpr int front_lds() {
  return max_c<max_c<km_partial_lds<D, NT>(), v_tiles_f16_lds<D>()>(), max_c<POOL ? psq_lds<128, D, NT>() : 16, POOL ? 16 : 4 * MASK_NKP_FRONT + 64>()>();
}

template <int D, int DT, bool POOL, int QR, int NT>
__global__ __launch_bounds__(NT) void front_kernel(const FrontParams p) {
  __shared__ __align__(16) unsigned char smem[front_lds<D, POOL, NT>()];
  const int w = blockIdx.x;
  if (w == 0 && threadIdx.x < 8 && (!POOL || p.nk > SPG_SELECT_IN_ATTN_NK)) p.queue[threadIdx.x] = 0;
  if (w >= p.wg_q) {
    const int id = w - p.wg_q, bh = id / p.nq;
    float thr = 0.f;
    if constexpr (POOL) thr = p.simthr.at(bh % p.H);
    psq_body<128, D, DT, MEAN_NONE, POOL, QR, NT>(p.q, p.qs, nullptr, nullptr, 0, p.pool_q, p.sim_q, p.q8, p.q_scale, thr, p.H, p.N, p.nq,
                                              id - bh * p.nq, bh, smem);
  } else if (w < p.wg_v) {
    const int bh = w / p.k_chunks;
    km_partial_body<D, DT, NT>(p.k, p.ks, p.Hkv, p.km_part, p.Nk, p.k_rows, w - bh * p.k_chunks, p.k_chunks, bh, smem);
  } else if (w < p.wg_mask) {
    const int id = w - p.wg_v;
    if (p.v_f16) {
      const int bh = id / p.nk;
      if (p.v_dtype == 0) v_tiles_f16_body<D, 0, NT>(p.v, p.vs, p.Hkv, p.v_tiles, p.Nk, p.nk, id - bh * p.nk, bh, smem);
      else v_tiles_f16_body<D, 1, NT>(p.v, p.vs, p.Hkv, p.v_tiles, p.Nk, p.nk, id - bh * p.nk, bh, smem);
    } else {
      const int bh = id / p.v_chunks;
      float *dst = p.v_part + (size_t)id * D;
      auto store = [&](int d, float s) { dst[d] = s; };
      if (p.v_dtype == 0) v_absmax_body<D, 0, NT>(p.v, p.vs, p.Hkv, p.Nk, p.v_rows, id - bh * p.v_chunks, bh, smem, store);
      else v_absmax_body<D, 1, NT>(p.v, p.vs, p.Hkv, p.Nk, p.v_rows, id - bh * p.v_chunks, bh, smem, store);
    }
  } else if constexpr (!POOL) {
    const size_t row = (size_t)(w - p.wg_mask);
#define SPG_M2L(K_) case K_: map_to_lut_body<K_, NT>(p.mask, p.lut, p.valid, p.nk, p.nkp, row, smem); break;
    switch (p.mask_kind) { SPG_M2L(0) SPG_M2L(1) SPG_M2L(2) SPG_M2L(3) SPG_M2L(4) SPG_M2L(5) SPG_M2L(6) }
#undef SPG_M2L
  }
}

struct FinalParams {
  const double *km_part;
  const float *v_part;
  uint16_t *km;
  float *v_amax;
  int k_chunks, v_chunks, N;            // v_chunks == 0: no V maxima
};

// blockDim = (D, 8): eight threads share a column's partial results
template <int D, int DT>
__global__ void final_kernel(const FinalParams p) {
  __shared__ double s_sub[8][D];
  __shared__ float s_max[8][D];
  const int bh = blockIdx.x, d = threadIdx.x, y = threadIdx.y;
  double s = 0.0;
#pragma unroll 4
  for (int i = y; i < p.k_chunks; i += 8) s += p.km_part[((size_t)bh * p.k_chunks + i) * D + d];
  float m = 0.f;
#pragma unroll 4
  for (int i = y; i < p.v_chunks; i += 8) m = fmaxf(m, p.v_part[((size_t)bh * p.v_chunks + i) * D + d]);
  s_sub[y][d] = s;
  s_max[y][d] = m;
  __syncthreads();
  if (y == 0) {
#pragma unroll
    for (int u = 1; u < 8; u++) { s += s_sub[u][d]; m = fmaxf(m, s_max[u][d]); }
    p.km[(size_t)bh * D + d] = f64_to_elem<DT>(s / (double)p.N);
    if (p.v_chunks > 0) p.v_amax[(size_t)bh * D + d] = m;
  }
}

// rows of K per workgroup of the back kernel
constexpr int k_rows_per_wg(int nt) { return nt == 256 ? 128 : 64; }

struct BackParams {
  const uint16_t *k, *v;
  Strides ks, vs;
  int H, Hkv, Nk, nk;                   // H: query heads (simthr has one entry per query head)
  int v_dtype;
  int wg_v;                             // workgroups below it quantise K, the others V
  int k_wgs_per_head;
  const uint16_t *km;
  const double *km_part;
  int k_chunks;
  const float *v_amax, *v_part;
  int v_chunks;
  uint16_t *v_tiles;                    // V16
  Hyper simthr;
  uint16_t *pool_k;
  uint8_t *sim_k;
  int8_t *k8;
  float *k_scale;
  uint8_t *v8;
  float *v_scale;
};

// PARTIAL: the partial results of the front kernel are combined here, by every workgroup for the head it works on
// V16: V goes to FP16 tiles (f16_tiles_in_back)
template <int D, int DT, bool POOL, bool PARTIAL, bool V16, int NT>
__global__ __launch_bounds__(NT) void back_kernel(const BackParams p) {
  constexpr int ROWS = k_rows_per_wg(NT);
  constexpr int LK = max_c<POOL ? psq_lds<64, D, NT, ROWS>() : 16, NT * 8 + 2 * D>();
  constexpr int LV = V16 ? v_tiles_f16_lds<D>() : v_quant_lds<D>() + 4 * NT + 4 * D;
  __shared__ __align__(16) unsigned char smem[max_c<LK, LV>()];
  const int w = blockIdx.x;
  if (w < p.wg_v) {
    const int bh = w / p.k_wgs_per_head;
    float thr = 0.f;
    if constexpr (POOL) thr = p.simthr.at((bh % p.Hkv) * (p.H / p.Hkv));
    psq_body<64, D, DT, PARTIAL ? MEAN_PARTIAL : MEAN_GIVEN, POOL, 64, NT, ROWS>(p.k, p.ks, p.km, p.km_part, p.k_chunks, p.pool_k, p.sim_k, p.k8,
                                                                  p.k_scale, thr, p.Hkv, p.Nk, p.nk, w - bh * p.k_wgs_per_head, bh, smem);
  } else if constexpr (V16) {
    const int id = w - p.wg_v, bh = id / p.nk, blk = id - bh * p.nk;
    if (p.v_dtype == 0) v_tiles_f16_body<D, 0, NT>(p.v, p.vs, p.Hkv, p.v_tiles, p.Nk, p.nk, blk, bh, smem);
    else v_tiles_f16_body<D, 1, NT>(p.v, p.vs, p.Hkv, p.v_tiles, p.Nk, p.nk, blk, bh, smem);
  } else {
    const int id = w - p.wg_v, bh = id / p.nk, blk = id - bh * p.nk;
    float *s_amax = (float *)(smem + v_quant_lds<D>());
    float *s_sub = s_amax + D;
    const int tid = threadIdx.x;
    if constexpr (PARTIAL) {
      float m = 0.f;
#pragma unroll 4
      for (int i = tid / D; i < p.v_chunks; i += NT / D) m = fmaxf(m, p.v_part[((size_t)bh * p.v_chunks + i) * D + tid % D]);
      s_sub[tid] = m;
      __syncthreads();
      if (tid < D) {
#pragma unroll
        for (int u = 1; u < NT / D; u++) m = fmaxf(m, s_sub[tid + u * D]);
        s_amax[tid] = m;
      }
    } else if (tid < D) {
      s_amax[tid] = p.v_amax[(size_t)bh * D + tid];
    }
    __syncthreads();
    if (blk == 0 && tid < D) p.v_scale[(size_t)bh * D + tid] = s_amax[tid] / 2.25f;
    auto amax_of = [&](int d) { return s_amax[d]; };
    if (p.v_dtype == 0) v_quant_body<D, 0, NT>(p.v, p.vs, p.Hkv, p.v8, p.Nk, p.nk, blk, bh, smem, amax_of);
    else v_quant_body<D, 1, NT>(p.v, p.vs, p.Hkv, p.v8, p.Nk, p.nk, blk, bh, smem, amax_of);
  }
}

// Short heads: front and back in one launch.  Every workgroup that quantises a block of K sums the columns of its whole head for
// itself, every one that quantises a block of V takes the maxima of its whole head; the rest are the front kernel's mask rows and Q
// blocks.  Bound by the chain of one workgroup - its head from L2 (at most 256 KiB), the sums, then the block - which is shorter than
// the two launches.
struct ShortParams {
  FrontParams f;
  BackParams b;
  int wg_v, wg_mask, wg_q;              // first workgroup of each role behind the blocks of K
};
template <int D, int DT, bool POOL, int QR>
__global__ __launch_bounds__(512) void short_kernel(const ShortParams p) {
  constexpr int NT = 512, ROWS = k_rows_per_wg(NT);
  constexpr int LK = max_c<POOL ? psq_lds<64, D, NT, ROWS>() : 16, NT / 64 * 128 * 8 + 2 * D>();
  constexpr int LV = max_c<max_c<v_quant_lds<D>(), v_absmax_lds<D, NT>()>() + 4 * D, v_tiles_f16_lds<D>()>();
  constexpr int LQ = max_c<POOL ? psq_lds<128, D, NT>() : 16, POOL ? 16 : 4 * MASK_NKP_FRONT + 64>();
  __shared__ __align__(16) unsigned char smem[max_c<max_c<LK, LV>(), LQ>()];
  const int w = blockIdx.x;
  const FrontParams &f = p.f;
  const BackParams &b = p.b;
  if (w == 0 && threadIdx.x < 8 && !POOL) f.queue[threadIdx.x] = 0;
  if (w < p.wg_v) {
    const int bh = w / b.k_wgs_per_head;
    float thr = 0.f;
    if constexpr (POOL) thr = b.simthr.at((bh % b.Hkv) * (b.H / b.Hkv));
    psq_body<64, D, DT, MEAN_HERE, POOL, 64, NT, ROWS>(b.k, b.ks, nullptr, nullptr, 0, b.pool_k, b.sim_k, b.k8, b.k_scale, thr, b.Hkv, b.Nk, b.nk,
                                                       w - bh * b.k_wgs_per_head, bh, smem);
  } else if (w < p.wg_mask) {
    const int id = w - p.wg_v, bh = id / b.nk, blk = id - bh * b.nk;
    if (f.v_f16) {
      if (b.v_dtype == 0) v_tiles_f16_body<D, 0, NT>(b.v, b.vs, b.Hkv, b.v_tiles, b.Nk, b.nk, blk, bh, smem);
      else v_tiles_f16_body<D, 1, NT>(b.v, b.vs, b.Hkv, b.v_tiles, b.Nk, b.nk, blk, bh, smem);
    } else {
      float *const s_amax = (float *)(smem + max_c<v_quant_lds<D>(), v_absmax_lds<D, NT>()>());
      auto store = [&](int d, float s) { s_amax[d] = s; };
      if (b.v_dtype == 0) v_absmax_body<D, 0, NT>(b.v, b.vs, b.Hkv, b.Nk, b.Nk, 0, bh, smem, store);
      else v_absmax_body<D, 1, NT>(b.v, b.vs, b.Hkv, b.Nk, b.Nk, 0, bh, smem, store);
      __syncthreads();
      if (blk == 0 && threadIdx.x < D) b.v_scale[(size_t)bh * D + threadIdx.x] = s_amax[threadIdx.x] / 2.25f;
      auto amax_of = [&](int d) { return s_amax[d]; };
      if (b.v_dtype == 0) v_quant_body<D, 0, NT>(b.v, b.vs, b.Hkv, b.v8, b.Nk, b.nk, blk, bh, smem, amax_of);
      else v_quant_body<D, 1, NT>(b.v, b.vs, b.Hkv, b.v8, b.Nk, b.nk, blk, bh, smem, amax_of);
    }
  } else if (w >= p.wg_q) {
    const int id = w - p.wg_q, bh = id / f.nq;
    float thr = 0.f;
    if constexpr (POOL) thr = f.simthr.at(bh % f.H);
    psq_body<128, D, DT, MEAN_NONE, POOL, QR, NT>(f.q, f.qs, nullptr, nullptr, 0, f.pool_q, f.sim_q, f.q8, f.q_scale, thr, f.H, f.N, f.nq,
                                                  id - bh * f.nq, bh, smem);
  } else if constexpr (!POOL) {
    const size_t row = (size_t)(w - p.wg_mask);
#define SPG_M2L(K_) case K_: map_to_lut_body<K_, NT>(f.mask, f.lut, f.valid, f.nk, f.nkp, row, smem); break;
    switch (f.mask_kind) { SPG_M2L(0) SPG_M2L(1) SPG_M2L(2) SPG_M2L(3) SPG_M2L(4) SPG_M2L(5) SPG_M2L(6) }
#undef SPG_M2L
  }
}
template <int D, int DT>
static void run_short(const spg_attn_args *a, const ShortParams &p, int wgs, hipStream_t st) {
  const bool pool = a->selection != SPG_SELECT_MASK;
  if constexpr (D == 128) {
    if (a->qk_quant_gran == SPG_QUANT_PER_WARP) {
      if (pool) short_kernel<D, DT, true, 32><<<wgs, 512, 0, st>>>(p);
      else short_kernel<D, DT, false, 32><<<wgs, 512, 0, st>>>(p);
      return;
    }
  }
  if (pool) short_kernel<D, DT, true, 128><<<wgs, 512, 0, st>>>(p);
  else short_kernel<D, DT, false, 128><<<wgs, 512, 0, st>>>(p);
}

template <int D, int DT, int NT>
static void run_front(bool pool, bool per_warp, const FrontParams &f, int wgs, hipStream_t st) {
  // (a pass of the workgroup stays inside one 32-row quantisation group: the wide form needs D = 128 for it)
  if constexpr (NT == 256 || D == 128) {
    if (per_warp) {
      if (pool) front_kernel<D, DT, true, 32, NT><<<wgs, NT, 0, st>>>(f);
      else front_kernel<D, DT, false, 32, NT><<<wgs, NT, 0, st>>>(f);
      return;
    }
  }
  if (pool) front_kernel<D, DT, true, 128, NT><<<wgs, NT, 0, st>>>(f);
  else front_kernel<D, DT, false, 128, NT><<<wgs, NT, 0, st>>>(f);
}
template <int D, int DT, int NT>
static void run_back(bool pool, bool partial, bool v16, const BackParams &b, int wgs, hipStream_t st) {
#define SPG_BACK(POOL_, PARTIAL_)                                                          \
  {                                                                                        \
    if (v16) back_kernel<D, DT, POOL_, PARTIAL_, true, NT><<<wgs, NT, 0, st>>>(b);          \
    else back_kernel<D, DT, POOL_, PARTIAL_, false, NT><<<wgs, NT, 0, st>>>(b);             \
  }
  if (partial) { if (pool) SPG_BACK(true, true) else SPG_BACK(false, true) }
  else         { if (pool) SPG_BACK(true, false) else SPG_BACK(false, false) }
#undef SPG_BACK
}
template <int D, int DT>
static void run_front_back(const spg_attn_args *a, const FrontParams &f, const BackParams &b, const Chunks &c, uint16_t *km, float *v_amax,
                           int front_nt, int front_wgs, int back_nt, int back_wgs, hipStream_t st) {
  const bool pool = a->selection != SPG_SELECT_MASK, per_warp = a->qk_quant_gran == SPG_QUANT_PER_WARP;
  if (front_nt == 512) run_front<D, DT, 512>(pool, per_warp, f, front_wgs, st);
  else run_front<D, DT, 256>(pool, per_warp, f, front_wgs, st);
  if (!c.partial) {
    const FinalParams p = {f.km_part, f.v_part, km, v_amax, f.k_chunks, a->pv_f16 ? 0 : f.v_chunks, a->N_kv};
    final_kernel<D, DT><<<a->B * a->Hkv, dim3(D, 8), 0, st>>>(p);
  }
  if (back_nt == 512) run_back<D, DT, 512>(pool, c.partial, f16_tiles_in_back(a), b, back_wgs, st);
  else run_back<D, DT, 256>(pool, c.partial, f16_tiles_in_back(a), b, back_wgs, st);
}

hipError_t run_forward(const spg_attn_args *a, const Strides &qs, const Strides &ks, const Strides &vs, const Strides &os,
                              hipStream_t st) {
  const Layout l = layout_for(a);
  unsigned char *ws = (unsigned char *)a->workspace;
  const int heads = a->B * a->H, kv_heads = a->B * a->Hkv;
  const int nq = (a->N + 127) / 128, nk = (a->N_kv + 63) / 64;
  const Chunks c = chunks_for(a);
  const bool pool = a->selection != SPG_SELECT_MASK;
  const Hyper simthr = {a->simthreshd1, a->simthreshd1_value};
  int32_t *const lut = (int32_t *)(ws + l.lut);
  int32_t *const valid = !pool && a->valid_block_num != nullptr ? a->valid_block_num : (int32_t *)(ws + l.valid);
  // Fewer than two workgroups of 256 threads per CU leave the stages bound by the length of one thread's work (9.8 and
  // 13.0 us for the two launches at B2 H3 N1025 D128 with a similarity threshold): twice the threads take half of it.
  const bool in_one = one_launch(a), sel_in_attn = pool && nk <= SPG_SELECT_IN_ATTN_NK, front_q = q_in_front(a) || q_overwritten(a, qs, os);
  const int q_wgs = front_q ? heads * nq : 0;
  const bool can_wide = !(a->D == 64 && a->qk_quant_gran == SPG_QUANT_PER_WARP);
  const bool tiles_in_back = f16_tiles_in_back(a);
  const int v_front = a->pv_f16 ? tiles_in_back ? 0 : kv_heads * nk : kv_heads * c.n;
  const int front_nt = in_one || (q_wgs + front_chunk_wgs(a) <= 512 && (can_wide || !front_q)) ? 512 : 256;
  const int back_nt = in_one || (heads * nq + kv_heads * 2 * c.n <= 512 && can_wide) ? 512 : 256;
  int nkp = 256;
  while (nkp < nk || nkp < front_nt) nkp <<= 1;
  const bool mask_in_front = !pool && nkp <= MASK_NKP_FRONT;

  FrontParams f = {};
  f.q = (const uint16_t *)a->q; f.k = (const uint16_t *)a->k; f.v = (const uint16_t *)a->v;
  f.qs = qs; f.ks = ks; f.vs = vs;
  f.H = a->H; f.Hkv = a->Hkv; f.N = a->N; f.Nk = a->N_kv; f.nq = nq; f.nk = nk;
  f.v_dtype = a->v_dtype; f.v_f16 = a->pv_f16;
  f.k_chunks = f.v_chunks = c.n; f.k_rows = f.v_rows = c.rows;
  f.wg_v = kv_heads * c.n;
  f.wg_mask = f.wg_v + v_front;
  f.wg_q = f.wg_mask + (mask_in_front ? heads * nq : 0);
  f.km_part = (double *)(ws + l.km_part); f.v_part = (float *)(ws + l.v_part); f.v_tiles = (uint16_t *)(ws + l.v);
  f.mask = a->mask; f.mask_kind = a->mask_kind; f.nkp = nkp; f.lut = lut; f.valid = valid;
  f.simthr = simthr;
  f.pool_q = (uint16_t *)(ws + l.pool_q); f.sim_q = ws + l.sim_q; f.q8 = (int8_t *)(ws + l.q8); f.q_scale = (float *)(ws + l.q_scale);
  f.queue = (int *)(ws + l.queue);

  BackParams b = {};
  b.k = f.k; b.v = f.v; b.ks = ks; b.vs = vs;
  b.H = a->H; b.Hkv = a->Hkv; b.Nk = a->N_kv; b.nk = nk; b.v_dtype = a->v_dtype;
  b.k_wgs_per_head = (a->N_kv + k_rows_per_wg(back_nt) - 1) / k_rows_per_wg(back_nt);
  b.wg_v = kv_heads * b.k_wgs_per_head;
  b.km = (const uint16_t *)(ws + l.km); b.km_part = f.km_part; b.k_chunks = c.n;
  b.v_amax = (const float *)(ws + l.v_amax); b.v_part = f.v_part; b.v_chunks = c.n;
  b.simthr = simthr;
  b.pool_k = (uint16_t *)(ws + l.pool_k); b.sim_k = ws + l.sim_k; b.k8 = (int8_t *)(ws + l.k8); b.k_scale = (float *)(ws + l.k_scale);
  b.v8 = ws + l.v; b.v_tiles = f.v_tiles; b.v_scale = (float *)(ws + l.v_scale);

  if (in_one) {
    ShortParams s = {f, b, 0, 0, 0};
    s.wg_v = b.wg_v;
    s.wg_mask = s.wg_v + kv_heads * nk;
    s.wg_q = s.wg_mask + (mask_in_front ? heads * nq : 0);
    const int wgs = s.wg_q + heads * nq;
    if (a->D == 64) { if (a->qk_dtype == 0) run_short<64, 0>(a, s, wgs, st); else run_short<64, 1>(a, s, wgs, st); }
    else            { if (a->qk_dtype == 0) run_short<128, 0>(a, s, wgs, st); else run_short<128, 1>(a, s, wgs, st); }
  } else {
    const int front_wgs = f.wg_q + q_wgs, back_wgs = b.wg_v + (a->pv_f16 && !tiles_in_back ? 0 : kv_heads * nk);
    uint16_t *km = (uint16_t *)(ws + l.km);
    float *v_amax = (float *)(ws + l.v_amax);
#define SPG_RUN(D_, DT_) run_front_back<D_, DT_>(a, f, b, c, km, v_amax, front_nt, front_wgs, back_nt, back_wgs, st)
    if (a->D == 64) { if (a->qk_dtype == 0) SPG_RUN(64, 0); else SPG_RUN(64, 1); }
    else            { if (a->qk_dtype == 0) SPG_RUN(128, 0); else SPG_RUN(128, 1); }
#undef SPG_RUN
  }
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  RowSelect sel = {};
  if (sel_in_attn)
    sel = {f.pool_q, b.pool_k, f.sim_q, b.sim_k, Hyper{a->level, a->level_value}, a->selection == SPG_SELECT_TOPK, a->is_causal,
           a->attention_sink, a->valid_block_num};
  else if (pool)
    e = launch_block_select_h(f.pool_q, f.sim_q, b.pool_k, b.sim_k, a->selection == SPG_SELECT_TOPK, Hyper{a->level, a->level_value},
                              a->is_causal, a->attention_sink, lut, valid, a->valid_block_num, nullptr, a->B, a->H, a->Hkv, nq, nk, a->D, a->qk_dtype, st);
  else if (!mask_in_front)
    e = launch_map_to_lut(a->mask, a->mask_kind, lut, valid, a->B, a->H, nq, nk, st);
  if (e != hipSuccess) return e;
  RowSplit split = {};
  if (rows_in_chunks(a)) split = row_split(chunk_plan(a->B, a->H, a->N, a->N_kv, a->D), ws + l.split);
  const RawQ raw = {f.q, qs, simthr};
  return launch_block_sparse_attn_h(f.q8, b.k8, b.v8, a->out, os, a->qk_dtype, lut, valid, sel_in_attn ? &sel : nullptr, front_q ? nullptr : &raw,
                                    Hyper{a->pvthreshd, a->pvthreshd_value},
                                    f.q_scale, b.k_scale, a->pv_f16 ? nullptr : b.v_scale, a->B, a->H, a->Hkv, a->N, a->N_kv, a->D,
                                    a->sm_scale, a->kernel_causal ? 1 : 0, a->qk_quant_gran == SPG_QUANT_PER_WARP ? 1 : 0,
                                    SPG_PV_PER_BLOCK, nullptr, pool && a->is_causal, f.queue, &split,
                                    front_q ? few_rows(a) : 0, st);
}

}  // namespace spg
