// kvc_prefill_split.h -- the rule for the work split of a prefill launch (host
// code without HIP, so that a test can compile it alone).
#pragma once

#include <algorithm>
#include <cmath>

#include "kvc_internal.h"

namespace kvc {

// Work split of a prefill launch: rows per workgroup (16 or 32) and key tiles
// per piece (0: groups are not split).  One workgroup runs per CU, so a launch
// of few workgroups, or of workgroups of very unequal lengths, takes as long as
// its longest one; 16-row workgroups are shorter, and cut into pieces a launch
// takes as long as its work spread over all CUs plus the fold of the pieces.
// Each choice is priced in us and the cheapest taken:
//  - whole workgroups, dispatched longest first, take whole rounds: as long as
//    the longest, as the rounds of the shortest, or as the work spread over the
//    CUs plus a share of what the longest has over the shortest.  A workgroup
//    is a fixed part (q, first tile, epilogue) and its tiles;
//  - pieces, many and of unequal lengths, cost a smaller fixed part (no
//    epilogue), the fold's launch, a partial written and read at 6 TB/s, and a
//    margin, since they slow each other once they fill the card (64 sequences
//    of 8 rows over 100-3000 keys: 116 us unsplit, 129 split).
// The constants of whole workgroups are fitted to kvc_prefill_attn and
// kvc_prefill_step with bf16 and fp32 rows at 134 batches of 1-64 sequences,
// 8-2000 rows and 0-16000 keys with either size: against the faster one the
// choice loses 0.9 % in the mean.  us per layer, 32-row / 16-row workgroups: 13
// sequences of 100 rows over none 17.0 / 21.9 (q given), 24.2 / 29.7 (bf16 rows),
// 28.6 / 33.4 (fp32 rows); 24 of 48 14.7 / 18.9, 22.6 / 27.7, 25.0 / 31.2; one
// of 500 24.4 / 19.0, 32.8 / 26.4, 34.8 / 27.5.
// kvc_prefill_step, us per layer, the former kernel (32 rows, never split) ->
// the choice made: 32 rows over 4001 keys 132.6 -> 26.8; 128 rows over 16000
// keys 489 -> 59; 128 rows over 1000 keys 47.2 -> 25.8; 500 rows over none 33.6
// -> 26.7 (16 rows, unsplit); 40 sequences of 16 rows over 100-12000 keys 368 ->
// 237.  Launches of 512 and more 32-row workgroups have no idle CU to fill.
inline void prefill_split(PrefillArgs& a) {
    constexpr double kCus = 256, kTail = 0.3, kFold = 6.0, kPartBytesPerUs = 6e6, kMargin = 1.15;
    const auto blocks_of = [&](int rows) { return (a.n_q + rows - 1) / (int64_t)rows; };
    a.rows = 32;
    a.piece_tiles = 0;
    if (a.n_groups * blocks_of(32) >= 2 * (int64_t)kCus) return;
    double best = 1e30;
    const auto take = [&](double cost, int rows, int64_t piece_tiles) {
        if (cost >= best) return;
        best = cost;
        a.rows = rows;
        a.piece_tiles = (int32_t)piece_tiles;
    };
    for (int rows = 16; rows <= 32; rows += 16) {
        const int64_t n_pb = blocks_of(rows);
        const auto tiles_of = [&](int32_t j, int64_t b) {
            return (a.q_pos0[j] + std::min<int64_t>((b + 1) * rows, a.n_q) + kPfKeys - 1) / kPfKeys;
        };
        int64_t total = 0, longest = 0, shortest = INT64_MAX;
        for (int32_t j = 0; j < a.n_seqs; j++)
            for (int64_t b = 0; b < n_pb; b++) {
                const int64_t t = tiles_of(j, b);
                total += t * kKvHeads;
                longest = std::max(longest, t);
                shortest = std::min(shortest, t);
            }
        {
            const double fixed = rows == 16 ? 8.0 : 10.0, tile = rows == 16 ? 1.7 : 1.75;
            const double most = fixed + tile * longest, least = fixed + tile * shortest;
            const double wgs = (double)(a.n_groups * n_pb);
            double cost = most;
            if (wgs > kCus)
                cost = std::max({most, std::ceil(wgs / kCus) * least,
                                 (wgs * fixed + tile * total) / kCus + kTail * (most - least)});
            take(cost, rows, 0);
        }
        const double fixed = rows == 16 ? 5.0 : 9.0, tile = rows == 16 ? 1.7 : 1.95;
        for (int64_t t = longest - std::max<int64_t>(1, longest / 5); t >= 1; t -= std::max<int64_t>(1, t / 5)) {
            int64_t wgs = 0, parts = 0, slots = 0;
            for (int32_t j = 0; j < a.n_seqs; j++) {
                slots += (tiles_of(j, n_pb - 1) + t - 1) / t * kKvHeads * n_pb;
                for (int64_t b = 0; b < n_pb; b++) {
                    const int64_t p = (tiles_of(j, b) + t - 1) / t * kKvHeads;
                    wgs += p;
                    if (p > kKvHeads) parts += p;
                }
            }
            if (slots > pf_max_parts(rows)) break;
            const double rounds = std::max(1.0, wgs / kCus);
            const double cost = rounds * fixed + tile * (wgs <= kCus ? t : std::max((double)t, total / kCus + 0.5 * t));
            take(kMargin * (cost + kFold + parts * pf_part_floats(rows) * 8 / kPartBytesPerUs), rows, t);
        }
    }
}

}  // namespace kvc
