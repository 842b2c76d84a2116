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
    int part_gaps;           // 1: the merge reads the partials of live splits only
    long long merge_wave0;   // the split merge's launch: its first wave
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

// A kernel form of one head dim: 16-query blocks per wave, stage halves or not, waves, and
// its cost in us: `wg` and `row` per workgroup and query row of it (Q and first-stage loads,
// the pipeline's fill, epilogue) and `stage` per 32-key stage.  Fitted, with the split's costs
// below, to graph-replayed times of 20,000 forced (form, split) plans of 1,830 chunks (1 .. 4096
// queries, past 0 .. 30,000, GQA 1 .. 16, K = V or not).  Of a chunk's forced plans the cheapest
// by this cost then takes 1.008 (D = 128), 1.004 (256) and 1.010 (512) times the fastest's time
// on average, 1.05, 1.03 and 1.06 at the 95th percentile, 1.20 at most.
struct Tiling {
    int qb, kh, nw;
    float wg, row, stage;
    int rows() const { return 16 * qb * (kh ? nw / 2 : nw); }
};

// The forms a head dim can run, tallest first.  At D = 256, 256-row tiles' two blocks a wave
// share each K and V read; 64-row tiles split their stages between the wave groups.  At D = 512
// a stage is bound by each wave's own chain, so four waves on 64 rows take nearly as long as
// eight on 128; but where CUs would idle, the smaller tiles halve what each loads and writes:
// 32 fresh tokens 15.9 -> 10.1 us, 100 18.6 -> 13.0, 16 over 5016 keys 32.4 -> 28.7, 20 over 973
// separate K / V rows 24.5 -> 21.3.
constexpr Tiling kTilings512[] = {{1, 0, 8, 5.7f, 0.076f, 1.54f}, {1, 0, 4, 6.2f, 0.066f, 1.6f}};
constexpr Tiling kTilings256[] = {{2, 0, 8, 5.47f, 0.033f, 1.7f}, {1, 0, 8, 4.94f, 0.036f, 1.014f},
                                  {1, 1, 8, 5.93f, 0.05f, 0.62f}};
constexpr Tiling kTilings128[] = {{2, 0, 8, 5.16f, 0.017f, 1.055f}};

constexpr int kXcds = 8, kEngines = 4, kEngineCus = kTargetGroups / (kXcds * kEngines);
constexpr float kEmptyUs = 1.0f;  // a workgroup whose split holds no key of its tile

// Estimated us until the last workgroup of a plan ends.  Whatever their lengths, workgroup i
// goes to XCD i % 8 and an XCD's workgroups in turn to its four engines of 8 CUs, each to the CU
// that falls idle first, none before the one ahead of it on the XCD.  With 2 (kv head, split)
// pairs a tile per XCD, or 1 of 4 or 8 in all, some engines or XCDs then get all the long
// workgroups: 2705 queries over 3739 keys at D = 128, 85 tiles of one head, take 89 us in 4
// splits and 62 in 3; 2043 fresh ones, 32 tiles of 8 heads, 77 unsplit and 100 in 2.  (Any CU
// of the GPU, or of the XCD, to the next workgroup: 52 and 73 us estimated for those two.)
// nst: stages of each tile, latest first; last_rows: query rows of the latest tile.
inline float makespan(const Tiling &t, const int *nst, int tiles, int last_rows, int Hkv, int splits, int per) {
    float ends[kXcds][kEngines][kEngineCus] = {}, front[kXcds] = {};
    float most = 0.0f;
    unsigned wg = 0;
    for (int i = 0; i < tiles; ++i)
        for (int s = 0; s < splits; ++s) {
            const int n = std::min(per, nst[i] - s * per);
            const float us = n > 0 ? t.wg + t.row * (i ? t.rows() : last_rows) + n * t.stage : kEmptyUs;
            for (int h = 0; h < Hkv; ++h, ++wg) {
                const unsigned xcd = wg % kXcds;
                float *e = ends[xcd][wg / kXcds % kEngines];
                unsigned cu = wg / (kXcds * kEngines);
                if (cu >= kEngineCus) {
                    cu = 0;
                    for (int c = 1; c < kEngineCus; ++c) cu = e[c] < e[cu] ? c : cu;
                    front[xcd] = std::max(front[xcd], e[cu]);
                }
                e[cu] = front[xcd] + us;
                most = std::max(most, e[cu]);
            }
        }
    return most;
}

// Splitting adds a dependent launch and D fp32 per row and split, written by the attention
// kernel and read by the merge.  Few partials are stored non-temporal: the merge reads them
// from other XCDs, and the launch boundary then has no dirty lines to write back (64 local
// queries in 4 splits, 8 MB: 19.5 -> 17.9 us; 200 in 2, 13 MB: 28.3 -> 25.2).  Past the XCDs'
// L2s together (8 x 4 MB) the write-back overlaps the kernel, and waiting for memory costs
// more: 32 MB 46.7 -> 45.7 us, 40 MB 43.7 both ways, 48 MB 42.2 -> 46.4, 64 MB 42.2 -> 54.0.
constexpr float kPartNtBytes = 36.0e6f;

// Where a quarter of the tiles have no key in the last split (the first ones: a tile sees more
// than those before it, up to the window), the merge first reads which splits of a row are
// live.  That second round trip costs few partials more than their empty ones do: fresh queries
// of 16 heads, D = 256, 8.4 MB (256 in 2 splits) 2.8 -> 3.1 us, 12.6 MB 3.2 -> 3.5, 16.8 MB
// 3.6 -> 3.6 .. 4.2, 25 MB 5.0 -> 4.9, 50 MB 9.0 -> 6.1.
constexpr float kGapBytes = 20.0e6f;
inline float split_cost(float part_bytes, int splits) {  // us
    // (the merge's forms: up to 4 splits, up to 8, more)
    return 3.2f + 2.2e-7f * part_bytes + (splits > 4 ? 0.3f : 0.0f) + (splits > 8 ? 0.9f + 0.11f * (splits - 8) : 0.0f);
}
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
    // rounds of 256 CUs: 333 queries over 5933 keys (K = V, 21 tiles of 4 heads) take 126 us as 252
    // workgroups and 190 as 336, whose second round is mostly idle.
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
            if (f) break;
            return "esda_prefill: too many query tiles";
        }
        const bool few = groups <= kMaxRounds * kTargetGroups;
        int nst[kMaxRounds * kTargetGroups];  // few: stages of each tile, latest first
        const int last_rows = (int) (rows - (tiles - 1) * QT);
        int most = 1, most_full = 0;  // stages of the longest tile, and of those of QT rows
        double total = 0.0;
        for (int i = 0; i < (int) tiles; ++i) {
            int a, b;
            tile_keys(*p, (int) tiles - 1 - i, QT, a, b);
            const int n = (int) (((long long) b - a + kStageKeys - 1) / kStageKeys);
            if (few) nst[i] = n;
            most = std::max(most, n);
            if (i || last_rows == QT) most_full = std::max(most_full, n);
            total += t.wg + t.row * (i ? QT : last_rows) + n * t.stage;
        }
        const float even = (float) (total * d->num_kv_heads / kTargetGroups);
        auto consider = [&](int per) {  // per: stages per split
            const int splits = (most + per - 1) / per;
            float us = splits > 1 ? split_cost(4.0f * D * (float) rows * d->num_kv_heads * splits, splits) : 0.0f;
            const float longest = std::max(t.wg + t.row * last_rows + std::min(per, most) * t.stage,
                                           most_full ? t.wg + t.row * QT + std::min(per, most_full) * t.stage : 0.0f);
            // no plan is faster than its longest workgroup, nor than its work spread evenly
            if (us + std::max(longest, even) >= best) return;
            if (groups * splits <= kTargetGroups) {
                us += longest;  // one round
            } else if (few && groups * splits <= 2LL * kMaxRounds * kTargetGroups) {
                // nor than its pieces' work spread evenly, nor the rounds that its whole pieces take
                int whole = 0, pieces = 0;
                for (int i = 0; i < (int) tiles; ++i) {
                    whole += nst[i] / per;
                    pieces += (nst[i] + per - 1) / per;
                }
                const int rounds = (whole * d->num_kv_heads + kTargetGroups - 1) / kTargetGroups;
                const float spread = even + (float) (pieces - tiles) * d->num_kv_heads * t.wg / kTargetGroups;
                if (us + std::max(spread, rounds * (t.wg + per * t.stage)) >= best) return;
                us += makespan(t, nst, (int) tiles, last_rows, d->num_kv_heads, splits, per);
            } else {
                // many workgroups (many tiles, or forced splits of any count): each piece starts anew, and
                // the CUs stay busy but for the end of the last round.  (70 chunks of forced splits that
                // took shorter tiles without the pieces' starts: 14% less time on average; 3028 queries
                // over 3787 keys in 4 splits, D = 256, 16 heads, 344 us in 128-row tiles, 229 in 256-row.)
                const double more = (double) tiles * (splits - 1) * d->num_kv_heads / kTargetGroups;
                us += even + (float) more * (t.wg + t.row * QT) + 0.5f * (t.wg + t.row * QT + std::min(per, most) * t.stage);
            }
            if (us < best) {
                best = us;
                kps = per * kStageKeys;
                most_stages = most;
                p->qb = t.qb;
                p->kh = t.kh;
                p->nw = t.nw;
                p->tiles = (int) tiles;
            }
        };
        if (d->split_keys > 0) {
            consider(d->split_keys / kStageKeys);
        } else {
            consider(most);
            int last = most;
            for (int s = 2; s <= most && groups * s <= kMaxRounds * kTargetGroups; s += std::max(1, s / 4)) {
                const int per = (most + s - 1) / s;
                if (per != last) consider(per);
                last = per;
            }
        }
        if (!few) break;  // many rounds of the tallest tiles: nothing for shorter ones to fill
    }
    if (d->split_keys > 0) kps = d->split_keys;
    const long long splits = ((long long) most_stages * kStageKeys + kps - 1) / kps;
    if (splits > 65535 || (long long) p->tiles * d->num_kv_heads * splits > INT_MAX)
        return "esda_prefill: too many key splits";
    p->kps = kps;
    p->splits = (int) std::max<long long>(1, splits);
    const float part_bytes = 4.0f * D * p->Sq * p->Hq * p->splits;
    p->part_nt = part_bytes <= kPartNtBytes;
    int a, b;
    tile_keys(*p, p->tiles / 4, 16 * p->qb * (p->kh ? p->nw / 2 : p->nw), a, b);
    p->part_gaps = part_bytes > kGapBytes && b - a <= (p->splits - 1) * (long long) p->kps;
    return nullptr;
}

// A launch of the split merge takes 2^31 threads (a HIP launch holds fewer than 2^32).  More rows
// take several.
constexpr long long kMergeLaunchWaves = 1LL << 25;
inline long long merge_waves(const PrefillParams &p, int D) {
    const long long rows = (long long) p.Sq * p.Hq;
    return D == 512 ? 2 * rows : D == 128 && p.splits <= 8 ? (rows + 1) / 2 : rows;
}

inline size_t workspace_of(const PrefillParams &p, int D) {
    if (p.splits <= 1) return 0;
    const size_t rows = (size_t) p.Sq * p.Hq;
    return (size_t) p.splits * rows * ((size_t) D * 4 + 8) + 256;
}

}  // namespace esda_prefill_plan
