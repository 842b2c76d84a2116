// prefill_plan_check.cpp -- the plan of esda_prefill (apertura_amd/csrc/esda_prefill_plan.h)
// for descriptions read from standard input, one per line: "Hq Hkv D Sq Sk q_pos0 k_pos0
// window split_keys".  Prints, per line, the kernel form and split (waves, query rows per
// tile, tiles per kv head, key splits, keys per split, whether the merge reads live splits
// only, workspace bytes), or the refusal.
// Built and run by tests/test_plan_arithmetic.py with g++.
#include "esda_prefill_plan.h"

#include <cstdio>

int main() {
    esda_prefill_desc d{};
    int n = 0;
    while (std::scanf("%d %d %d %d %d %d %d %d %d", &d.num_q_heads, &d.num_kv_heads, &d.head_dim, &d.seq_q, &d.seq_k,
                      &d.q_pos0, &d.k_pos0, &d.window, &d.split_keys) == 9) {
        d.q_head_stride = (int64_t) d.seq_q * d.head_dim;
        d.q_row_stride = d.head_dim;
        d.kv_head_stride = (int64_t) d.seq_k * d.head_dim;
        d.out_row_stride = (int64_t) d.num_q_heads * d.head_dim;
        d.out_head_stride = d.head_dim;
        d.scale = 1.0f;
        esda_prefill_plan::PrefillParams p;
        if (const char *why = esda_prefill_plan::plan_prefill(&d, &p)) std::printf("refused: %s\n", why);
        else
            std::printf("%d %d %d %d %d %d %zu\n", p.nw, 16 * p.qb * (p.kh ? p.nw / 2 : p.nw), p.tiles, p.splits, p.kps,
                        p.part_gaps, esda_prefill_plan::workspace_of(p, d.head_dim));
        ++n;
    }
    return n == 0;
}
