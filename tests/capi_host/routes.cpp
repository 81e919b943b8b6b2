// Prints the route of whole-operator calls, one line per call read from standard input:
//   B H Hkv N N_kv D selection pv_f16 simthreshd1 level is_causal pvthreshd
//     ->  one_launch chunks combined_by_the_back_kernel groups_per_row q_in_front workspace_bytes chunks_of_a_row_at_most rows_in_chunks few_rows some_level_in_chunks
// The rules are host code (spargeattn_amd/csrc/forward_plan.h); nothing is launched.
#include "forward_plan.h"

#include <cstdio>

int main() {
  spg_attn_args a = {};
  a.qk_quant_gran = SPG_QUANT_PER_BLOCK;
  while (std::scanf("%d %d %d %d %d %d %d %d %f %f %d %f", &a.B, &a.H, &a.Hkv, &a.N, &a.N_kv, &a.D, &a.selection, &a.pv_f16, &a.simthreshd1_value, &a.level_value, &a.is_causal, &a.pvthreshd_value) == 12) {
    const spg::Chunks c = spg::chunks_for(&a);
    std::printf("%d %d %d %d %d %zu %d %d %d %d\n", (int)spg::short_heads(&a), c.n, (int)c.partial,
                spg::attn_groups(a.B * a.H * ((a.N + 127) / 128), (a.N_kv + 63) / 64, a.D, a.pv_f16 != 0), (int)spg::q_in_front(&a), spg::layout_for(&a).total, spg::chunk_plan(a.B, a.H, a.N, a.N_kv, a.D).chunks, (int)spg::rows_in_chunks(&a), spg::few_rows(&a), (int)spg::may_have_rows_in_chunks(&a));
  }
  return 0;
}
