// esda_prefill_plan.h -- how a prefill call is laid out: the kernel parameters, the keys a
// query tile sees, the kernel form (tile height, waves) and the key splits of a description,
// and the workspace they need.  esda_prefill.hip plans and launches with it;
// tests/prefill_plan_check.cpp compiles it with g++ and prints the plan of any description.
#pragma once

#include <algorithm>
#include <climits>
#include <cmath>
#include <cstddef>
#include <cstdint>

#include "esda_plan.h"
#include "esda_prefill.h"

namespace esda_prefill_plan {

constexpr int kStageKeys = 32;
constexpr int kTargetGroups = 256;         // one workgroup per CU

struct PrefillParams {
    const uint16_t *q, *k, *v;
    uint16_t *out;
    float *part_acc;   // [splits][Sq * Hq][D]
    float *part_ml;    // [splits][Sq * Hq][2]
    long long q_hs, q_rs, kv_hs, o_rs, o_hs;
    int Hq, Hkv, G, Sq, Sk, q_pos0, k_pos0, window;
    int qb;                  // 16-query blocks per wave
    int tiles, splits, kps;  // query tiles per kv head, key splits, keys per split
    float scale_log2e;
    int kh;                  // 1: the two wave groups split each tile's stages (even / odd)
    int nw;                  // waves per workgroup (query tile: 16 qb nw rows, half of it with kh)
    int part_nt;             // 1: partials stored non-temporal
};

// Query row r of a GQA group's rows -> its position in the chunk (r % G is its head).  At
// most 2^24 tiles of 256 rows (plan_prefill), so 32-bit divisions: the 64-bit ones took
// ~4,000 of a workgroup's first 13,000 cycles.
ESDA_HD unsigned position_of(long long r, int G) { return (unsigned) r / (unsigned) G; }

// Keys [j0, j1) that some row of query tile `tile` (QT rows) can see.
ESDA_HD void tile_keys(const PrefillParams &p, int tile, int QT, int &j0, int &j1) {
    const long long rows = (long long) p.Sq * p.G;
    const long long r0 = (long long) tile * QT;
    const long long r1 = (r0 + QT < rows ? r0 + QT : rows) - 1;
    const long long qa0 = p.q_pos0 + position_of(r0, p.G), qa1 = p.q_pos0 + position_of(r1, p.G);
    long long lo = p.window > 0 ? qa0 - p.window + 1 - p.k_pos0 : 0;
    long long hi = qa1 - p.k_pos0 + 1;
    if (lo < 0) lo = 0;
    if (hi > p.Sk) hi = p.Sk;
    if (hi < lo) hi = lo;
    j0 = (int) lo;
    j1 = (int) hi;
}

// A kernel form of one head dim: 16-query blocks per wave, stage halves or not, and its
// cost in us with one workgroup per CU: `wg` per workgroup (Q and first-stage loads, the
// pipeline's fill, epilogue) and `stage` per 32-key stage.  Fitted to graph-replayed times
// over 1 .. 470 stages and 4 .. 512 workgroups; the plans then lie within 5% of the best
// forced split on 40 of 45 random chunks (the others within 14%).
struct Tiling {
    int qb, kh, nw;
    float wg, stage;
    int rows() const { return 16 * qb * (kh ? nw / 2 : nw); }
};

// The forms a head dim can run.  At D = 256, per 32 keys: 64-row stage-halves tiles 0.66 us,
// 128-row tiles 1.16, and 256-row tiles, whose two blocks share each K and V read, 1.9.  At D =
// 512 a stage is bound by each wave's own chain, so four waves on 64 rows take nearly as long
// as eight on 128; but where CUs would idle, the smaller tiles halve what each loads and
// writes: 32 fresh tokens 15.9 -> 10.1 us, 100 18.6 -> 13.0, 16 over 5016 keys 32.4 -> 28.7, 20 over
// 973 separate K / V rows 24.5 -> 21.3.
constexpr Tiling kTilings512[] = {{1, 0, 4, 5.5f, 1.38f}, {1, 0, 8, 9.0f, 1.5f}};
constexpr Tiling kTilings256[] = {{1, 1, 8, 5.5f, 0.66f}, {1, 0, 8, 5.5f, 1.16f}, {2, 0, 8, 8.0f, 1.9f}};
constexpr Tiling kTilings128[] = {{2, 0, 8, 3.5f, 1.0f}};

// Estimated us of a plan: `pieces(f)` calls f(stages) for each workgroup of one kv head in
// dispatch order.  The heads run side by side, so one head has kTargetGroups / Hkv CUs; the
// dispatcher hands a workgroup to the CU that falls idle first, which for the descending
// lengths of the tiles (latest first) is the order back and forth over the CUs.
template <class F>
float makespan(int Hkv, const Tiling &t, F &&pieces) {
    const int cus = std::max(1, kTargetGroups / Hkv);
    const float share = Hkv > kTargetGroups ? (float) Hkv / kTargetGroups : 1.0f;  // heads per CU
    float load[kTargetGroups];
    std::fill_n(load, cus, 0.0f);
    int at = 0, dir = 1;
    pieces([&](int stages) {
        load[at] += t.wg + stages * t.stage;
        if (at + dir < 0 || at + dir >= cus) dir = -dir;  // the end takes two in a row
        else at += dir;
    });
    float most = 0.0f;
    for (int i = 0; i < cus; ++i) most = std::max(most, load[i]);
    return most * share;
}

// Splitting adds a dependent launch and D fp32 per row and split, written by the attention
// kernel and read by the merge.  Few partials are stored non-temporal: the merge reads them
// from other XCDs, and the launch boundary then has no dirty lines to write back (64 local
// queries in 4 splits, 8 MB: 19.5 -> 17.9 us; 200 in 2, 13 MB: 28.3 -> 25.2).  Past the XCDs'
// L2s together (8 x 4 MB) the write-back overlaps the kernel, and waiting for memory costs
// more: 32 MB 46.7 -> 45.7 us, 40 MB 43.7 both ways, 48 MB 42.2 -> 46.4, 64 MB 42.2 -> 54.0.
constexpr float kPartNtBytes = 36.0e6f;
inline float split_cost(float part_bytes) { return 5.0f + 3.1e-7f * part_bytes; }  // us
constexpr int kMaxRounds = 3;  // split plans of more workgroups per CU only add partials

// Validates a description and fills the kernel parameters' shape fields and plan.  Returns
// what is wrong with it, or null.
inline const char *plan_prefill(const esda_prefill_desc *d, PrefillParams *p) {
    if (!d) return "esda_prefill: null description";
    const int D = d->head_dim;
    if (D != 128 && D != 256 && D != 512)
        return "esda_prefill: head_dim must be 128, 256 or 512";
    if (d->num_q_heads <= 0 || d->num_kv_heads <= 0 || d->num_q_heads % d->num_kv_heads)
        return "esda_prefill: num_q_heads must be a multiple of num_kv_heads";
    if (d->seq_q <= 0 || d->seq_k <= 0 || d->window < 0 || d->q_pos0 < 0 || d->k_pos0 < 0)
        return "esda_prefill: sizes, positions and window must be non-negative";
    if ((long long) d->q_pos0 + d->seq_q > INT_MAX || (long long) d->k_pos0 + d->seq_k > INT_MAX)
        return "esda_prefill: positions must stay below 2^31";
    if (d->k_pos0 > d->q_pos0 || (long long) d->k_pos0 + d->seq_k < (long long) d->q_pos0 + d->seq_q)
        return "esda_prefill: the keys must hold every query's own position (k_pos0 <= q_pos0, "
                    "k_pos0 + seq_k >= q_pos0 + seq_q)";
    for (long long st : {d->q_head_stride, d->q_row_stride, d->kv_head_stride, d->out_row_stride, d->out_head_stride})
        if (st < 0 || st % 8)
            return "esda_prefill: strides must be non-negative multiples of 8";
    if (d->kv_head_stride < (long long) d->seq_k * D && d->num_kv_heads > 1)
        return "esda_prefill: kv_head_stride smaller than a head's rows";
    if (d->split_keys < 0 || d->split_keys % kStageKeys)
        return "esda_prefill: split_keys must be a multiple of 32";
    if (!(d->scale > 0.0f) || !std::isfinite(d->scale))
        return "esda_prefill: scale must be positive and finite";
    *p = PrefillParams{};
    p->Hq = d->num_q_heads;
    p->Hkv = d->num_kv_heads;
    p->G = d->num_q_heads / d->num_kv_heads;
    p->Sq = d->seq_q;
    p->Sk = d->seq_k;
    p->q_pos0 = d->q_pos0;
    p->k_pos0 = d->k_pos0;
    p->window = d->window;
    p->q_hs = d->q_head_stride;
    p->q_rs = d->q_row_stride;
    p->kv_hs = d->kv_head_stride;
    p->o_rs = d->out_row_stride;
    p->o_hs = d->out_head_stride;
    p->scale_log2e = d->scale * 1.4426950408889634f;
    // Form and split: the cheapest by the cost above.  What counts is how the workgroups fill
    // rounds of 256 CUs: 333 queries over 5933 keys (84 tiles) take 135 us as 252 workgroups
    // and 192 us as 336, whose second round is mostly idle; 770 fresh tokens (192 tiles) 51 us
    // unsplit and 80 us split in two.
    const long long rows = (long long) d->seq_q * p->G;
    const Tiling *forms = D == 512 ? kTilings512 : D == 256 ? kTilings256 : kTilings128;
    const int nforms = D == 512 ? 2 : D == 256 ? 3 : 1;
    float best = INFINITY;
    int kps = 0, most_stages = 0;  // of the best plan
    for (int f = 0; f < nforms; ++f) {
        const Tiling &t = forms[f];
        const int QT = t.rows();
        const long long tiles = (rows + QT - 1) / QT, groups = tiles * d->num_kv_heads;
        if (groups > (1LL << 24)) {
            if (f + 1 < nforms) continue;
            return "esda_prefill: too many query tiles";
        }
        const bool few = groups <= kMaxRounds * kTargetGroups;
        int nst[kMaxRounds * kTargetGroups];  // few: stages of each tile, latest first
        int most = 1;
        double total = 0.0;
        for (int i = 0; i < (int) tiles; ++i) {
            int a, b;
            tile_keys(*p, (int) tiles - 1 - i, QT, a, b);
            const int n = (int) (((long long) b - a + kStageKeys - 1) / kStageKeys);
            if (few) nst[i] = n;
            most = std::max(most, n);
            total += t.wg + n * t.stage;
        }
        auto consider = [&](int per) {  // per: stages per split
            const int splits = (most + per - 1) / per;
            float us = splits > 1 ? split_cost(4.0f * D * (float) rows * d->num_kv_heads * splits) : 0.0f;
            // no plan is faster than its longest workgroup, nor than its work spread evenly
            if (us + std::max(t.wg + std::min(per, most) * t.stage,
                              (float) (total * d->num_kv_heads / kTargetGroups)) >= best)
                return splits;
            if (few && tiles * splits <= 2LL * kMaxRounds * kTargetGroups)
                us += makespan(d->num_kv_heads, t, [&](auto &&piece) {
                    for (int i = 0; i < (int) tiles; ++i)
                        for (int j = 0; j < nst[i]; j += per) piece(std::min(per, nst[i] - j));
                });
            else  // many workgroups: the CUs stay busy but for the end of the last round
                us += (float) (total * d->num_kv_heads / kTargetGroups) + 0.5f * (t.wg + most * t.stage);
            if (us < best) {
                best = us;
                kps = per * kStageKeys;
                most_stages = most;
                p->qb = t.qb;
                p->kh = t.kh;
                p->nw = t.nw;
                p->tiles = (int) tiles;
            }
            return splits;
        };
        if (d->split_keys > 0) {
            consider(d->split_keys / kStageKeys);
        } else {
            consider(most);
            for (int s = 2; s <= most && groups * s <= kMaxRounds * kTargetGroups;)
                s = std::max(s, consider((most + s - 1) / s)) + std::max(1, s / 4);
        }
    }
    if (d->split_keys > 0) kps = d->split_keys;
    const long long splits = ((long long) most_stages * kStageKeys + kps - 1) / kps;
    if (splits > 65535 || (long long) p->tiles * d->num_kv_heads * splits > INT_MAX)
        return "esda_prefill: too many key splits";
    p->kps = kps;
    p->splits = (int) std::max<long long>(1, splits);
    p->part_nt = 4.0f * D * p->Sq * p->Hq * p->splits <= kPartNtBytes;
    return nullptr;
}

inline size_t workspace_of(const PrefillParams &p, int D) {
    if (p.splits <= 1) return 0;
    const size_t rows = (size_t) p.Sq * p.Hq;
    return (size_t) p.splits * rows * ((size_t) D * 4 + 8) + 256;
}

}  // namespace esda_prefill_plan
