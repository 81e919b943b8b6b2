// Host side of the whole-operator call, free of device code: which launches it takes, how the partial sums are split, where
// everything lies in the workspace.  Shared by the entry points (capi.hip) and the launches (forward.hip).
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
// Many heads: sixteen chunks each already spread the read over the chip.  What takes its time then is a chunk of N / 16 rows, which
// needs something beside it, and the reading of sixteen chunks by every workgroup of the back kernel, which grows with all rows of
// K.  At D = 128 that something is a front grid large enough for 256 threads per workgroup (more than 512 workgroups; below, the chunks
// are all there is) and the gain ends early; a mask takes the work of pooling off the blocks of Q, and with it what the chunks hide
// behind.  At D = 64, half the bytes in a row, it is 512 blocks of Q (1280 for fewer than sixteen heads), or none over short heads.
// us per call with sixteen chunks / with the final kernel, top-k 0.4, heads x queries x keys (steady runs over three sets of inputs;
// calls of the two forms in turn mislead here, their workspaces differ):
// D128 16 x 1024 x 8200 92 / 97, 12 x 4096 x 12288 151 / 156, 16 x 256 x 16384 145 / 148, 24 x 4096 x 8200 175 / 176, 12 x 8192 186 / 189, 32 x 1024 x
// 8200 124 / 126; 12 x 1024 x 8200 89 / 85, 12 x 256 x 32768 265 / 243, 10 x 1024 x 16384 140 / 132, 48 x 1024 x 16384 314 / 309, 24 x 16384 883 / 878;
// masks 16 x 1024 x 8200 94 / 90, 12 x 16384 468 / 455, 24 x 4096 x 16384 306 / 295, 48 x 16384 1770 / 1756.
// D64 48 x 256 x 8200 94 / 96, 24 x 4096 x 8200 118 / 122, 24 x 12288 359 / 372, 16 x 16384 405 / 422, 24 x 4096 x 20480 252 / 258, 16 x 8192 x 32768
// 429 / 440, 12 x 20480 475 / 490; 16 x 1024 x 12288 90 / 87, 12 x 4096 x 16384 149 / 143, 10 x 256 x 32768 187 / 164, 24 x 1024 x 32768 226 / 220, 32 x
// 4096 x 32768 486 / 480, 48 x 20480 equal; masks 16 x 16384 412 / 441, 12 x 20480 471 / 500, 32 x 4096 x 8200 150 / 158, 16 x 1024 x 32768 187 / 182.
struct Chunks {
  int n, rows;
  bool partial;
};
inline Chunks chunks_for(const spg_attn_args *a) {
  Chunks c;
  const int N = a->N_kv, heads = a->B * a->Hkv;
  const long long all = (long long)heads * N, q_blocks = (long long)a->B * a->H * ((a->N + 127) / 128);
  const bool few = all <= 24576 && (long long)N * a->D < 3 << 19;
  const bool many = a->D == 128 ? a->selection != SPG_SELECT_MASK && heads >= 12 && q_blocks + 32ll * heads > 512 && all <= 294912
                                : (heads >= 16 && N <= 9216) || (heads >= 12 && q_blocks >= (heads >= 16 ? 512 : 1280) && N <= 32768 && all <= 786432);
  c.partial = N <= 8192 || few || many;
  const int want = N <= 8192 || many ? 16 : few ? 32 : (2048 + heads - 1) / heads;
  const int most = N <= 8192 ? (N + 63) / 64 : (N + 255) / 256;
  c.n = want < most ? want : most;
  c.rows = (N + c.n - 1) / c.n;
  c.n = (N + c.rows - 1) / c.rows;      // no chunk without rows
  return c;
}

// One launch instead of front and back (short_kernel): a workgroup reads its whole head, so the head has to be short, and all of
// them together read it once per block.  us per call with two launches / one, top-k H x N: D64 16 x 512 18.7 / 15.5, 2 x 1024 21.2 /
// 18.1, 8 x 1024 21.8 / 19.0, 2 x 1500 30.0 / 28.9, 1 x 2048 25.4 / 24.4, 1 x 2500 38.2 / 38.7, 40 x 400 22.3 / 22.8; D128 8 x 128 18.3 /
// 14.1, 8 x 512 22.2 / 18.8, 4 x 1024 25.2 / 23.9, 2 x 1200 32.2 / 31.7, 1 x 1500 35.5 / 36.0, 12 x 640 24.1 / 21.9, 30 x 512 25.8 / 27.0, 16 x
// 1024 30.6 / 34.7.  FP16 PV, whose V^T tiles need no maxima: D128 30 x 512 27.1 / 23.8, 16 x 1024 32.0 / 28.5, 40 x 400 30.7 / 26.6, 2 x 1500
// 38.0 / 38.7.  With a similarity threshold, whose work on a block outweighs the sums: D128 8 x 700 33.3 / 28.2, 20 x 700 41.1 / 38.5, 2 x
// 1500 40.1 / 38.0, 1 x 2048 45.1 / 44.6.
// Many queries over short heads: beyond about 1024 Q blocks the blocks of Q are most of the launch, and those go faster through the
// front kernel's 256 threads than through 512.  H, Nk, Q blocks: D128 8 x 512 1024 46.8 / 43.4, 24 x 512 768 40.3 / 40.5, 1536 58.6 / 60.5,
// 6144 172.6 / 183.5, 40 x 256 1280 47.0 / 45.8, 2560 72.2 / 73.9; D64 16 x 512 1024 35.5 / 32.6, 2048 50.8 / 52.7, 36 x 400 1152 42.9 / 42.5, 4608
// 92.5 / 106.0; FP16 PV 16 x 1024 1024 62.1 / 61.4, 30 x 512 1920 73.0 / 75.3; similarity 8 x 700 1024 76.1 / 72.1, 20 x 700 1280 88.3 / 89.2.
inline bool short_heads(const spg_attn_args *a) {
  const long long nq = (a->N + 127) / 128, nk = (a->N_kv + 63) / 64, kv_heads = (long long)a->B * a->Hkv;
  const long long head = (long long)a->N_kv * a->D, all = head * kv_heads * nk;
  const bool sim = a->selection != SPG_SELECT_MASK && (a->simthreshd1 != nullptr || a->simthreshd1_value >= 0.f);
  return head <= (sim ? 262144 : 155648) && all <= (a->pv_f16 ? 34 << 20 : sim ? 20 << 20 : 12 << 20) &&
         kv_heads * nk <= (a->pv_f16 ? 320 : 256) && (long long)a->B * a->H * nq <= 1024;
}

// (a pass of 512 threads over 64 channels covers two 32-row groups of Q scales)
inline bool one_launch(const spg_attn_args *a) { return !(a->D == 64 && a->qk_quant_gran == SPG_QUANT_PER_WARP) && short_heads(a); }

// FP16 PV: where V's tiles are written.  They depend on nothing and are bound by memory.  In the back kernel they stand beside blocks of K, which
// are bound by their vector instructions, and the front kernel is left with the sums of K; with no more blocks than CUs (of 128
// channels) both kernels are chains of latencies, and only the front one has places free under it.  us per call in front / in the back
// kernel, H x N (x Nk): D128 8 x 4096 CDF with similarity 92.0 / 88.2, 20 x 3840 103.8 / 99.5, 30 x 4096 x 1000 64.8 / 63.6, 40 x 700 41.1 / 39.8, 12 x
// 1024 x 8000 89.2 / 87.5, 32 x 1024 x 8200 138.0 / 133.7, 24 x 8192 causal 304.4 / 302.5, 24 x 16384 755.3 / 753.1; 1 x 2500 49.4 / 49.9, 2 x 4096 45.35
// / 45.46, 2 x 300 x 8000 121.3 / 121.6.  D64 30 x 8192 292.3 / 290.8, 16 x 1024 x 12288 95.7 / 93.9, 32 x 4096 x 8200 equal; 4 x 6000 71.9 / 72.2.
inline bool f16_tiles_in_back(const spg_attn_args *a) {
  return a->pv_f16 && (long long)a->B * a->Hkv * ((a->N_kv + 63) / 64) * a->D > 256 * 128 && !one_launch(a);
}

// Heads of K and V that the front kernel reads in chunks, and the workgroups that this takes.  Up to 512 of them, blocks of Q among them,
// have 512 threads each.
inline long long front_chunk_heads(const spg_attn_args *a) { return (long long)a->B * a->Hkv * (f16_tiles_in_back(a) ? 1 : 2); }
inline long long front_chunk_wgs(const spg_attn_args *a) { return front_chunk_heads(a) * chunks_for(a).n; }

// Whether Q is quantised (and pooled) in front of the attention kernel, or in place by its workgroups.  In place Q is read once, its codes never
// reach memory (half of Q's bytes written and read again), and the front kernel is left with K and V; but a row starts some 3 us later
// and its vector instructions are taken from the loops beside it.  That pays at D = 128 (twice the work per row of the list at the same
// cost) once rows beside each other cover the start.  us per call in front / in place, H x N (x Nk), two processes a side in turn:
// * with a selection from about two rows per CU, with a similarity threshold or without (of 144 shapes of 588 to 1300 rows and 400 to 2500 keys
//   each, top-k gains 2.0 % on average, CDF with similarity 1.4, FP16 PV 2.1; the largest losses are 2 %, just past the 768 rows that the chip holds at
//   once, 2.6 % with 400 keys).  Top-k 0.5: 10 x 5760 89.9 / 93.0, 16 x 4096 76.4 / 77.3, 20 x 3840 91.9 / 89.2, 40 x 2048 70.4 / 68.3, 80 x 1024 61.5 / 59.8, 24 x
//   4096 causal 97.5 / 93.9, 128 x 1024 83.0 / 82.5, 40 x 2560 x 700 53.7 / 54.6; CDF with similarity 16 x 3584 109.2 / 112.0, 10 x 8192 251 / 253, 20 x 3840 146.4 /
//   144.1, 24 x 4096 170 / 165, 20 x 5120 239.5 / 240.7, 32 x 8000 686 / 681, 40 x 2048 106.8 / 102.3, 24 x 8192 x 1000 115.9 / 111.9, 48 x 2176 x 400 67.5 / 69.3;
//   FP16 PV 80 x 1024 61.0 / 57.5, 20 x 3840 99.7 / 99.1, 16 x 8192 causal 217.2 / 214.4.
// * with a caller's mask, which needs no pooling, from 352 rows, if what is left to the front kernel is few enough workgroups to have 512 threads
//   each, which is most of that gain: 5 x 7680 82.8 / 85.8, 7 x 6528 83.3 / 80.8, 7 x 8192 99.3 / 94.2, 10 x 5120 74.6 / 72.8, 14 x 3712 63.9 / 63.8, 14 x
//   5248 89.3 / 85.2, GQA 32/8 x 1664 41.8 / 39.7, 28/4 x 2304 47.8 / 45.3.
// * with a mask and more heads of K, once the front kernel is bound by what it reads, from about 50 MB of Q, K and V (in a smaller one Q is
//   quantised beside chains of sums that take as long without it) and 480 rows: 20 x 2560 54.4 / 57.4, 28 x 2048 52.4 / 53.7, 36 x 2048 60.8 / 61.2, 48 x 1024
//   42.3 / 43.9, 80 x 640 39.8 / 41.8, 20 x 3712 77.3 / 77.5, 28 x 2944 73.6 / 72.5, 60 x 2048 85.8 / 82.2, 80 x 1024 57.9 / 55.7, 48 x 16384 1342 / 1318; 28 x 2688 x 1000
//   43.1 / 45.7, 36 x 2048 x 800 40.7 / 43.2, 44 x 2048 x 500 37.6 / 38.8, 22 x 4608 x 800 43.0 / 45.3, 28 x 3712 x 1500 57.9 / 57.8, 44 x 2944 x 800 54.9 / 53.9, 36 x 4608 x 1500
//   76.2 / 71.2, 48 x 16384 x 1000 193.4 / 177.9; 7 x 6528 x 12000 119.0 / 120.6, 7 x 9344 x 12000 equal.  Of 377 masks the rule is 0.1 % on average behind
//   the better side of each; 352 rows for all of them were 1 % and up to 7 %.
// D = 64: 14 x 6400 95.5 / 96.5, 22 x 6400 140.2 / 143.3, 30 x 8192 265.6 / 266.4, CDF 40 x 8000 585 / 605; masks 12 x 7500 83.9 / 84.8, 20 x 10240 124.1 /
// 125.7, 16 x 16384 325.7 / 325.3, 48 x 16384 657 / 650.  Where a selection kernel wants Q pooled, the front kernel reads Q anyway: H32 N32768
// causal 3953 / 3952, H30 N17776 D64 1007 / 1012.
inline bool q_in_front(const spg_attn_args *a) {
  const long long rows = (long long)a->B * a->H * ((a->N + 127) / 128);
  if (a->D == 64 || one_launch(a)) return true;
  if (a->selection != SPG_SELECT_MASK) return a->N_kv > 64 * SPG_SELECT_IN_ATTN_NK || rows <= 576;
  if (front_chunk_wgs(a) <= 512) return rows <= 352;
  return rows <= 480 || rows * 128 + front_chunk_heads(a) * a->N_kv <= 196608;   // (16-bit rows of 128 channels)
}

// In place a workgroup reads its Q block when others have stored their output already: `out` may be q itself, row on row, or lie apart.
inline bool q_overwritten(const spg_attn_args *a, const Strides &qs, const Strides &os) {
  if (a->q == a->out && qs.sb == os.sb && qs.sh == os.sh && qs.sn == os.sn) return false;
  auto bytes = [&](const Strides &s) { return (uintptr_t)(2 * ((a->B - 1) * s.sb + (a->H - 1) * s.sh + (a->N - 1) * s.sn + a->D)); };
  const uintptr_t q = (uintptr_t)a->q, out = (uintptr_t)a->out;
  return q < out + bytes(os) && out < q + bytes(qs);
}

// ---- rows in chunks (RowSplit) --------------------------------------------------------------------------------------
// Blocks of a chunk, and where the scratch for it lies.
//
// Up to 256 rows: about two rounds of workgroups if every block is kept (D = 64 fits four to a CU, D = 128 three), so that one
// round or more is left with half of them.  us per call by workgroups in all:
//                                       512   768  1024  1536  2048
//   D64   one head N17776, top-k 0.5    117   109    98    97   105
//         10000 x 10000, two heads       80    79    81    75    83
//   D128  one head N17776, top-k 0.5    160   140   133   140   143
//         the same, all blocks kept     186   194   191   194   197
//         10000 x 10000, two heads      106   101    96   103   108
// At least 16 blocks: 8300 x 8300 with 8 / 16 / 24 of them D64 55.5 / 53.4 / 57.6, D128 68.5 / 67.7 / 74.5.
//
// Beyond 256 rows: only for the sake of a partial last Q block, whose rows keep everything.  Beyond 1200 they would have two chunks
// (H12 N17776 top-k 0.15, 1668 rows, workgroup per row / chunks: D64 263 / 275, D128 351 / 391).  us by workgroups in all, N17776:
//                      1536  3072  4608                           1536  3072  4608
//   D64  H2 0.5         141   144   149      D128  H2 0.5          216   205   214
//        H4 0.15        143   129   132            H4 0.15         179   149   176
//        H4 0.3         167   180   171            H4 0.3          215   235   249
//        H4 0.5         247   223   233            H6 0.15         283   222   205
//        H8 0.15        218   185   171            N30001 H4 0.15  430   340   324
struct ChunkPlan {
  int chunks, per;                  // 1, 0: a row has one workgroup, whatever it keeps
  size_t first, maxima, md, o, bytes;
};
inline ChunkPlan chunk_plan(int B, int H, int N, int N_kv, int D) {
  ChunkPlan c = {1, 0, 0, 0, 0, 0, 0};
  const long long rows = (long long)B * H * ((N + 127) / 128), nk = (N_kv + 63) / 64;
  if (rows > (N % 128 != 0 ? 1200 : 256) || nk <= 36 || nk > 32768) return c;
  const long long wgs = rows > 256 ? 3072 : D == 64 ? 1536 : 1024, spread = (rows * nk + wgs - 1) / wgs;
  const long long most = (nk + 63) / 64;                          // 64 chunks: those of a row are added up one by one
  c.per = (int)(spread > most ? spread : most);
  if (c.per < 16) c.per = 16;
  c.chunks = (int)((nk + c.per - 1) / c.per);
  auto take = [&](size_t bytes) { const size_t r = c.bytes; c.bytes += (bytes + 255) / 256 * 256; return r; };
  const size_t all = (size_t)rows * c.chunks;                     // at most 4092, 275 MB at D = 128, whatever the lengths
  c.first = take(all * 4);
  c.maxima = take(all * 128 * 4);
  c.md = take(all * 256 * 4);
  c.o = take(all * 128 * D * 4);
  return c;
}
inline RowSplit row_split(const ChunkPlan &c, void *scratch) {
  unsigned char *const at = (unsigned char *)scratch;
  return {c.chunks, c.per, 0, (int *)(at + c.first), (float *)(at + c.maxima), (float *)(at + c.md), (float *)(at + c.o)};
}

// The share of a head's blocks that the chunks' time goes by.  A causal row keeps the smaller of `share` and what lies in front of the diagonal; an
// XCD works on an eighth of all rows, one behind the other, so with few heads the one with the last, longest rows of a head ends
// last: everything kept, a causal call takes 0.93, 0.83, 0.76 and 0.59 of the time that it takes without the diagonal with 1, 2, 4 and 8 heads (D64, 31950 and
// 17776 queries).
inline float blocks_that_count(long long heads, float share, bool causal) {
  if (!causal) return share;
  const float mean = share - 0.5f * share * share, part = heads < 8 ? heads / 8.f : 1.f, from = 1.f - part;      // rows from .. 1 of a head
  const float last = share <= from ? share : (0.5f * (share * share - from * from) + share * (1.f - share)) / part;
  return 0.3f * mean + 0.7f * last;
}

// Everything kept, with a partial last Q block: the longest row is as long as ever and the chunks have the most to do, so they pay nowhere
// less.  A workgroup per row takes 0.48 (D = 64), 0.62 (D = 128) and 0.74 us (FP16 PV) per block of a row in groups, and 0.9 and 1.1 us in one
// group beyond 256 rows; causal rows, half as many blocks, save a tenth of the chunks' time only (blocks_that_count).  us per call, workgroup per
// row / chunks, on both sides of the line, rows x nk:
//            up to 256 rows                                              beyond
// D64        188 x 376 215 / 192, 204 x 407 231 / 222, 252 x 251 156 / 185   376 x 376 375 / 339, 417 x 278 291 / 297, 390 x 130 157 / 166
// causal     219 x 438 241 / 231, 235 x 469 257 / 260, 252 x 251 154 / 160   417 x 278 256 / 236, 556 x 278 283 / 283, 469 x 938 819 / 830
// D128       157 x 313 242 / 218, 172 x 344 262 / 262, 204 x 407 300 / 348   278 x 278 359 / 336, 298 x 297 380 / 374, 376 x 376 465 / 518
// causal     172 x 344 258 / 237, 188 x 376 274 / 269, 204 x 407 293 / 317   298 x 297 338 / 312, 330 x 329 372 / 358, 417 x 278 320 / 346
// FP16 D64   172 x 344 206 / 190, 188 x 376 224 / 219, 204 x 407 238 / 245   376 x 376 396 / 379, 417 x 278 307 / 333, 470 x 469 487 / 574
// FP16 D128  157 x 313 288 / 252, 172 x 344 314 / 303, 204 x 407 362 / 405   266 x 532 712 / 651, 278 x 278 400 / 398, 298 x 297 425 / 440
inline bool chunks_pay_with_all_kept(int rows, int nk, int D, bool pv_f16, bool causal) {
  const float all = (float)rows * nk * (causal ? 0.9f : 1.f);
  if (rows > 256) return nk - all / (D == 64 ? 420.f : pv_f16 ? 290.f : 320.f) > 27.f;
  return nk - all / (D == 128 ? 185.f : pv_f16 ? 200.f : 220.f) > 36.f;
}

// Whether chunks pay: with a workgroup per row the call takes as long as its longest row, 0.45 us per block at D = 64 and 0.6 at D = 128
// (0.76 with FP16 PV); in chunks all blocks count, 2.05, 3.25 and 4.2 ns each, and the two launches more take 16 us.
//
// What a row keeps:
// * top-k without similar blocks to look for: what top-k names (share), and all of it in a partial last Q block, which is never similar.
//   simthreshd1: blocks of Q and K whose similarity is below it keep everything.  A similarity is not negative, so below 0 it changes nothing.
// * a similarity threshold of 0 or more, a CDF threshold or a level per head (share below 0): nothing on the host says.
//   With a partial last Q block the longest row keeps everything, and the chunks have the less to do the less the others keep: they have to pay with
//   everything kept.  us per call, workgroup per row / chunks, where they do not: H8 N17776 top-k 0.15 with simthreshd1 0.6, no block similar, D64 578 /
//   661, D128 831 / 1041; CDF 0.93 at 0.3, causal, one head N31595 D128 342 / 438; 0.82 at 0.6 N31887 with FP16 PV 457 / 531.
//   Whole rows with a top-k level keep that or more, and the more they keep the better for chunks, so it has to pay at the level (causal: without
//   the diagonal).
//   Whole rows without one keep anything, and a few of their blocks are one or two chunks: up to 64 rows of 288 K blocks or more, where what
//   is lost at low CDF thresholds is a tenth, and from 0.13 to 0.2 on there is a gain up to threefold.  One head, CDF threshold (no similarity test):
//                          0.02       0.06       0.09       0.13       0.2        0.35                   0.02       0.06       0.09       0.13       0.2        0.35
//     D64  8 x 288         31 / 33    36 / 41    41 / 44    46 / 44    55 / 48    76 / 49   D128         38 / 40    45 / 51    51 / 55    58 / 55    71 / 58    98 / 60
//          64 x 288        36 / 38    42 / 47    47 / 51    52 / 52    61 / 55    81 / 62                43 / 46    52 / 58    59 / 63    65 / 69    78 / 66   103 / 78
//          8 x 1000        59 / 63    77 / 69    91 / 69   110 / 71   142 / 73   211 / 80                69 / 74    94 / 80   113 / 81   138 / 84   180 / 86   267 / 89
//          64 x 200        32 / 33    36 / 40    40 / 44    44 / 48    50 / 49    64 / 56                37 / 39    44 / 47    48 / 53    54 / 58    62 / 60    81 / 68
//          100 x 256       34 / 36    40 / 44    43 / 48    48 / 52    57 / 59    74 / 65                40 / 42    48 / 54    54 / 61    60 / 64    71 / 74    94 / 83
//     one head, causal: N9088 D128 0.13 40 / 52, 0.2 46 / 53; N24064 D128 0.13 72 / 86, 0.2 88 / 116; not causal: N16000 D64 0.09 41 / 53
// * a mask: never in chunks.  Its density is known on the device only, and the rows of a sparse one are one or two chunks each, for which the
//   launches more cost up to a fifth of the call.  rows x nk, density:
//                  0.03          0.06          0.1           0.2                        0.03          0.06          0.1           0.2
//     D64  8 x 512   31.4 / 38.4   41.5 / 39.1   53.2 / 41.0   84.9 / 43.0    D128  8 x 512   41.6 / 49.0   54.9 / 49.8   70.5 / 52.2  112.4 / 55.0
//          64 x 256  31.6 / 36.2   38.1 / 43.2   45.5 / 44.8   60.1 / 50.0          64 x 256  45.0 / 50.2   54.3 / 59.5   62.9 / 60.4   81.5 / 65.3
//          64 x 288  39.8 / 43.8   48.0 / 52.8   58.2 / 53.7   74.1 / 58.3          64 x 288  59.5 / 63.9   68.4 / 76.4   80.9 / 78.1  100.6 / 82.4
//
// Up to 256 rows, top-k, us per call, workgroup per row / chunks, whole rows x nk:
//   D64   8 x 132    0.2  46.5 / 48.9, 0.35  56.0 / 51.9, 1.0  95.8 / 54.4    128 x 192  0.35 76.2 / 74.6, 0.5  90.4 / 82.0
//         64 x 132  0.35  59.9 / 57.8                                         128 x 512  0.2 115.5 / 113.5, 1.0 303 / 218
//         64 x 288   0.2  80.5 / 72.1, 1.0 183 / 111                          176 x 288  0.35 100 / 105, 1.0 182 / 175
//                                                                             224 x 512  1.0 321 / 332
//   D128  8 x 132    0.2  58.5 / 63.6, 0.35  72.3 / 66.8                      128 x 288  0.35 134 / 132, 0.5 161 / 143
//         64 x 512   0.1 128.7 / 133.4, 0.5 251 / 169                         176 x 512  1.0 405 / 423
//   FP16 PV, D128  64 x 288 0.2 107.5 / 95.3, 160 x 288 0.5 184 / 175, 256 x 288 0.5 198 / 217
// and with a partial last Q block, top-k 0.5: N24000, 188 rows, D64 207 / 145, causal 207 / 140, D128 265 / 190; N28000 D128 310 / 231; one head
// N17776 D64 CDF 171 / 136.
//
// Beyond 256 rows, where a row walks its blocks in one group, 0.7 us per block at D = 64 and 0.9 at D = 128, beside others or alone at the
// end; a partial last Q block, top-k:
//   N17776 D64   H2 0.15 231 / 96, 0.5 230 / 147, 0.7 243 / 180    H4 0.3 237 / 181, 0.5 254 / 227, 0.7 296 / 299    H6 0.3 243 / 229, 0.5 303 / 307
//                H8 0.15 246 / 186, 0.3 249 / 236    causal 0.5 H2 230 / 138, H4 250 / 218, H8 293 / 317    FP16 PV H2 0.5 243 / 152
//   N17776 D128  H2 0.15 276 / 113, 0.5 279 / 207    H3 0.3 283 / 200, 0.7 301 / 347    H4 0.3 303 / 239, 0.5 323 / 337    H8 0.15 326 / 278, 0.3 354 / 366
//                causal 0.5 H2 276 / 196, H4 308 / 322    FP16 PV H2 0.5 326 / 241
//   N8300 H6     0.15 D64 125 / 80, D128 154 / 107    0.5 D64 127 / 117, D128 156 / 161
//   30000 queries over 8400, two heads, 0.15  D64 119 / 66, D128 145 / 84
//   CDF 0.9 on N(0, 1) data, D64  H2 N17776 268 / 208, H4 338 / 342, H6 N8300 146 / 157
//
// Causal, us per call, workgroup per row / chunks, rows x nk, top-k 0.35, 0.6 and 1.0 (* the rule takes chunks):
//                    D64                                    D128                                   FP16 PV, D128
//   125 x 250         72 / 67   101 / 82*  143 / 100*         92 / 88   130 / 107* 187 / 146*       104 / 91   151 / 119* 223 / 165*
//   175 x 350         93 / 94   132 / 130  191 / 158*        118 / 129  170 / 171  247 / 234*       135 / 145  200 / 196  300 / 274*
//   200 x 400        103 / 109  147 / 138  214 / 191*        130 / 145  189 / 236  276 / 298        150 / 162  224 / 274  337 / 347
//   256 x 512        122 / 137  179 / 186  264 / 294         156 / 187  233 / 266  342 / 439        192 / 213  295 / 322  438 / 515
//   2 heads, 250     77 / 87    107 / 112  149 / 161          97 / 115  136 / 153  193 / 237        113 / 125  162 / 178  232 / 279
//   and with a partial last Q block
//   250 x 500        263 / 174* 263 / 230* 260 / 289         334 / 249* 334 / 345  335 / 442        418 / 282* 425 / 404* 431 / 516
//   H4 N17776        238 / 189* 266 / 251* 279 / 286         299 / 257* 328 / 347  346 / 427        357 / 298* 386 / 415  410 / 514
// Of 1800 calls, up to 1200 rows and 1000 K blocks, the rule is 0.3 % on average behind the better side; the worst that it cuts loses 2.2 %.
inline bool rows_in_chunks(int B, int H, int N, int N_kv, int D, bool pv_f16, int selection, float share, float simthreshd1, bool causal) {
  const int nk = (N_kv + 63) / 64, nq = (N + 127) / 128;
  if (selection == SPG_SELECT_MASK || nk <= SPG_SELECT_IN_ATTN_NK) return false;
  const ChunkPlan plan = chunk_plan(B, H, N, N_kv, D);
  if (plan.chunks == 1) return false;
  const bool many = B * H * nq > 256, partial = N % 128 != 0;
  const bool known = selection == SPG_SELECT_TOPK && share >= 0.f && simthreshd1 < 0.f;
  if (!known) {
    if (partial) return chunks_pay_with_all_kept(B * H * nq, nk, D, pv_f16, causal);
    if (share < 0.f) return B * H * nq <= 64 && nk >= 288;
    causal = false;
  }
  if (share > 1.f) share = 1.f;
  const float kept = share * nk;
  const float longest = partial ? (float)nk : kept;
  if (longest <= plan.per) return false;                            // no row has two chunks
  const float all = (float)(B * H) * (nq * nk * blocks_that_count((long long)B * H, share, causal) + (partial ? nk - kept : 0.f));
  if (many) return longest - all / (D == 64 ? 380.f : 250.f) > (D == 64 ? 56.f : 34.f);
  return longest - all / (D == 64 ? 190.f : partial && !pv_f16 ? 145.f : 170.f) > (D == 64 ? 34.f : 30.f);
}
inline bool rows_in_chunks(const spg_attn_args *a, float share, float simthreshd1) {
  return rows_in_chunks(a->B, a->H, a->N, a->N_kv, a->D, a->pv_f16 != 0, a->selection, share, simthreshd1, a->is_causal != 0);
}
// Whether some call of this shape with these options is cut.  The workspace has the scratch then, whatever hyper-parameters the call brings, and not
// otherwise: up to 275 MB beside some 50 (H8 N17776 D128).  For top-k the difference at the rule is linear in the share, or convex where it is
// causal, so it is largest at an end; a similarity threshold or a level per head only takes calls out.
inline bool may_have_rows_in_chunks(const spg_attn_args *a) {
  return a->selection == SPG_SELECT_TOPK ? rows_in_chunks(a, 0.f, -1.f) || rows_in_chunks(a, 1.f, -1.f) : rows_in_chunks(a, -1.f, 0.f);
}
inline bool rows_in_chunks(const spg_attn_args *a) {
  const float share = a->selection == SPG_SELECT_TOPK && a->level == nullptr ? (a->level_value > 0.f ? a->level_value : 0.f) : -1.f;
  // (without scratch never, however the sums at the line are rounded)
  return may_have_rows_in_chunks(a) && rows_in_chunks(a, share, a->simthreshd1 == nullptr ? a->simthreshd1_value : 0.f);
}

// Few short rows: workgroups to a row (few_rows_attn_kernel), or 0 where it has one.  Four while each has a CU to itself, two up to 128
// rows; the workgroup with all four quarters (attn_groups) beyond, and where a row has no more blocks than it has groups.  us per call, top-k
// 0.2, 0.5 and 1.0, rows x nk, one / four workgroups to a row:
//   D64   16 x 8    14.3 / 13.7   14.9 / 14.0   17.0 / 13.8       D128  16 x 4    14.5 / 14.8   15.5 / 14.6   16.6 / 14.2
//         64 x 16   16.4 / 14.4   19.0 / 15.3   22.3 / 16.0             64 x 16   22.5 / 19.9   26.3 / 21.6   30.6 / 23.4
//         64 x 64   26.5 / 22.0   37.1 / 26.9   53.4 / 32.8             64 x 128  54.2 / 42.7   78.6 / 55.5  116.8 / 73.7
//         64 x 128  44.0 / 34.5   61.9 / 43.5   90.4 / 57.0       FP16  64 x 64   36.4 / 30.6   52.7 / 41.7   76.4 / 54.5
//         96 x 16   16.5 / 19.5   19.2 / 21.5   22.6 / 23.1       (at D128)
// one / two:
//   D64   128 x 8   13.6 / 13.7   15.2 / 14.5   17.3 / 14.8       D128  128 x 8   16.7 / 17.6   19.7 / 18.6   22.3 / 20.0
//         128 x 16  16.6 / 15.8   19.3 / 17.2   22.6 / 19.5             128 x 16  23.1 / 22.2   26.7 / 24.7   31.5 / 28.3
//         128 x 128 45.2 / 40.2   62.5 / 55.3   91.6 / 78.5             128 x 128 54.3 / 49.5   78.8 / 68.2  116.5 / 99.0
//         160 x 32  21.5 / 27.9   27.5 / 34.5   34.5 / 45.7       FP16  128 x 64  38.0 / 37.5   53.9 / 54.1   77.4 / 77.6
// (FP16 PV at D128: its tiles leave room for three groups.)
//
// The workgroups of a row do not see each other's votes on the PV threshold.  A block is skipped when all scores of the Q block are `pvthreshd`
// below the running maxima in the exponent of 2; the quarter (half) of a workgroup alone may be that far below where the others are not, and
// then skips a block that the row keeps.  So the threshold has to be one at which that changes next to nothing: from 45 on, P of such a
// block is zero in e4m3 and in fp16, so O stays as it is (a product with an infinity or a NaN in V apart), and what is left out of a query's
// denominator is at most 64 x 2^-45 = 2^-39 of it per block, 2^-32 for 126 of them, below the rounding of its sum in binary32.
// (A per-head threshold is not known here: 0.)
inline int few_rows(int B, int H, int N, int N_kv, int D, bool pv_f16, float pvthreshd) {
  const long long rows = (long long)B * H * ((N + 127) / 128), nk = (N_kv + 63) / 64;
  if (!(pvthreshd >= 45.f) || nk > 128) return 0;
  if (rows <= 64) return nk >= 6 ? 4 : 0;
  return rows <= 128 && nk >= 12 && !(pv_f16 && D == 128) ? 2 : 0;
}
inline int few_rows(const spg_attn_args *a) {
  return few_rows(a->B, a->H, a->N, a->N_kv, a->D, a->pv_f16 != 0, a->pvthreshd == nullptr ? a->pvthreshd_value : 0.f);
}

struct Layout {
  size_t km_part, v_part, km, v_amax, pool_q, pool_k, sim_q, sim_k, q8, k8, q_scale, k_scale, v, v_scale, lut, valid, queue, split, total;
};
inline Layout layout_for(const spg_attn_args *a) {
  Layout l;
  size_t at = 0;
  auto take = [&](size_t bytes) { const size_t r = at; at += (bytes + 255) / 256 * 256; return r; };
  const size_t bh = (size_t)a->B * a->H, bhk = (size_t)a->B * a->Hkv, D = a->D;
  const size_t nq = ((size_t)a->N + 127) / 128, nk = ((size_t)a->N_kv + 63) / 64;
  const Chunks c = chunks_for(a);
  const bool pool = a->selection != SPG_SELECT_MASK;
  // (the parts that an attention kernel which quantises Q itself does not use are there all the same: the size follows from shapes and options
  // alone, whatever hyper-parameters a later call on the same workspace brings)
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
  l.split = take(may_have_rows_in_chunks(a) ? chunk_plan(a->B, a->H, a->N, a->N_kv, a->D).bytes : 0);
  l.total = at;
  return l;
}

// launches on `st`; the arguments have been checked
hipError_t run_forward(const spg_attn_args *a, const Strides &qs, const Strides &ks, const Strides &vs, const Strides &os, hipStream_t st);

}  // namespace spg
