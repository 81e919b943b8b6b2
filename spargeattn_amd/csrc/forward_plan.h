// Host side of the whole-operator call, free of device code: how the partial sums are split, where everything lies in the
// workspace.  Shared by the entry points (capi.hip) and the launches (forward.hip).
#pragma once
#include "../../include/spargeattn_amd.h"
#include "launch.h"

namespace spg {

// ---- workspace ----------------------------------------------------------------------------------------------------
// Partial column sums / maxima: `chunks` workgroups per head.  Up to 8192 rows a head has at most sixteen chunks, few
// enough to be combined by every workgroup of the back kernel (a few KiB from L2 against a launch of about 4.5 us);
// beyond, the final kernel combines as many as it takes to spread the read over the chip - unless the heads are so few that
// the back kernel's workgroups can read 32 chunks each for less than the launch (up to 24576 rows in all: at most 768
// workgroups, 13 MB from L2 in one head N17776 D64) and a head so short that reading its 32 chunks does not become the
// length of the front kernel (below 3 MiB of K).  us per call without / with the final kernel: one head D64 N12288 55.2 / 57.2,
// N17776 166.4 / 168.9, N20480 83.8 / 84.4, N24000 215.1 / 215.2, N24576 97.0 / 96.0; D128 N8448 59.9 / 61.5, N11000 145.8 / 146.9,
// N12000 157.9 / 157.8, N16384 94.6 / 93.5, N24576 132.0 / 126.3; two heads D128 N12288 80.9 / 80.9, with FP16 PV 88.9 / 88.3.
// Many heads: sixteen chunks each already spread the read over the chip, and the rest of the front kernel (Q, and the other
// heads) is long enough to hide that a chunk of up to 2048 rows takes its time - from about ten heads on, whatever N is.  us per call
// with / without the final kernel: 30 heads D64 N17776 1031 / 1026, 48 heads N16384 908 / 891, 32 heads N10000 425 / 408, 10 heads N24000
// 661 / 658; D128 12 heads N12000 385 / 380, 24 heads N9000 386.8 / 385.4, 32 heads N32768 causal 3913 / 3905; but 8 heads D64 N12000 193 /
// 202, 6 heads D128 N16384 288 / 290.
struct Chunks {
  int n, rows;
  bool partial;
};
inline Chunks chunks_for(int heads, int N, int D) {
  Chunks c;
  const bool few = (long long)heads * N <= 24576 && (long long)N * D < 3 << 19;
  const bool many = heads >= 12 && N <= 32768;
  c.partial = N <= 8192 || few || many;
  const int want = N <= 8192 || many ? 16 : few ? 32 : (2048 + heads - 1) / heads;
  const int most = N <= 8192 ? (N + 63) / 64 : (N + 255) / 256;
  c.n = want < most ? want : most;
  c.rows = (N + c.n - 1) / c.n;
  c.n = (N + c.rows - 1) / c.rows;      // no chunk without rows
  return c;
}

struct Layout {
  size_t km_part, v_part, km, v_amax, pool_q, pool_k, sim_q, sim_k, q8, k8, q_scale, k_scale, v, v_scale, lut, valid, queue, total;
};
inline Layout layout_for(const spg_attn_args *a) {
  Layout l;
  size_t at = 0;
  auto take = [&](size_t bytes) { const size_t r = at; at += (bytes + 255) / 256 * 256; return r; };
  const size_t bh = (size_t)a->B * a->H, bhk = (size_t)a->B * a->Hkv, D = a->D;
  const size_t nq = ((size_t)a->N + 127) / 128, nk = ((size_t)a->N_kv + 63) / 64;
  const Chunks c = chunks_for((int)bhk, a->N_kv, a->D);
  const bool pool = a->selection != SPG_SELECT_MASK;
  l.km_part = take(bhk * c.n * D * 8);
  l.v_part = take(a->pv_f16 ? 0 : bhk * c.n * D * 4);
  l.km = take(bhk * D * 2);
  l.v_amax = take(bhk * D * 4);
  l.pool_q = take(pool ? bh * nq * D * 2 : 0);
  l.pool_k = take(pool ? bhk * nk * D * 2 : 0);
  l.sim_q = take(pool ? bh * nq : 0);
  l.sim_k = take(pool ? bhk * nk : 0);
  l.q8 = take(bh * a->N * D);
  l.k8 = take(bhk * a->N_kv * D);
  l.q_scale = take(bh * nq * 4 * (a->qk_quant_gran == SPG_QUANT_PER_WARP ? 4 : 1));
  l.k_scale = take(bhk * nk * 4);
  l.v = take(bhk * nk * 64 * D * (a->pv_f16 ? 2 : 1));
  l.v_scale = take(bhk * D * 4);
  l.lut = take(bh * nq * nk * 4);
  l.valid = take(bh * nq * 4);
  l.queue = take(8 * sizeof(int));
  l.total = at;
  return l;
}

// launches on `st`; the arguments have been checked
hipError_t run_forward(const spg_attn_args *a, const Strides &qs, const Strides &ks, const Strides &vs, const Strides &os, hipStream_t st);

}  // namespace spg
