// kvc_decode_split.h -- the rule for the work split of a decode launch (host
// code without HIP, so that a test can compile it alone).
#pragma once

#include <algorithm>
#include <cmath>

#include "kvc_internal.h"

namespace kvc {

// Blocks per split-K chunk when the caller leaves it open, from the sequences'
// block counts nb[n].  Two ways to cut a launch:
//  - one workgroup per CU (at most 64 chunks x 4 heads, 32 chunks per
//    sequence for a short combine): the CUs share HBM, so it takes the time of
//    its bytes plus what the longest chunk has over the mean, at 0.45 us per
//    block of a workgroup alone;
//  - short chunks in many rounds, which balance ragged sequences: an item costs
//    7 ns of the launch's time, the last one of a CU 0.45 us per block, least
//    at 0.25 sqrt(total blocks) per chunk (lengths around it scatter by 2 %).
// The cheaper by that estimate is taken.  us per layer of kvc_decode_step, the
// former rule (4-block chunks, more only past 4096 items) -> this one: 1
// sequence of 300 tokens 7.74 -> 6.51, 2000 8.11 -> 7.39, 4200 10.35 -> 9.21,
// 32768 38.0 -> 27.3; 64 of 300 27.9 -> 19.0; 64 of 1000 59.6 -> 45.5; 8 of
// 777-6001 33.0 -> 26.3; kvc_decode_attn of 64 of 512-32768 (short chunks,
// fewer than before) 723 -> 703.
inline int32_t auto_chunk_blocks(const int32_t* nb, int32_t n, bool force_split) {
    int64_t total = 0;
    int32_t longest = 1;
    for (int32_t j = 0; j < n; j++) {
        total += nb[j];
        longest = std::max(longest, nb[j]);
    }
    // a chunk per sequence needs no exchange: 64 tokens 5.6 us, in two chunks
    // 6.4; 13 sequences of 4 blocks 7.81, in chunks of two 8.00, 48 of 97-128
    // tokens at most 10.41 against 10.78 (few of 4 blocks do better in chunks of
    // one: 1 sequence 6.34 against 6.55, 6 7.26 against 7.29)
    if (longest <= 3) return 3;
    if (longest == 4 && n >= 8) return 4;
    const auto chunks = [&](int32_t cb) {
        int64_t c = 0;
        for (int32_t j = 0; j < n; j++) c += (nb[j] + cb - 1) / cb;
        return c;
    };
    // smallest length with at most max_chunks chunks (monotone in it)
    const auto fit = [&](int32_t max_chunks) {
        int32_t lo = std::max<int32_t>((longest + 31) / 32, (int32_t)((total + max_chunks - 1) / max_chunks));
        int32_t hi = longest;
        while (lo < hi) {
            const int32_t mid = (lo + hi) / 2;
            if (chunks(mid) <= max_chunks)
                hi = mid;
            else
                lo = mid + 1;
        }
        return lo;
    };
    // short launches do better with two output-dim parts per chunk (up to 32
    // chunks) than with twice the chunks: 2 sequences of 1000 tokens 7.6 us
    // against 8.3; past 64 blocks where the longest sequence would have more
    // than 16 chunks to combine: 2 of 2048 tokens 8.5 us against 9.2 (32 chunks
    // each), 3 of 1200 8.6 against 9.0 (19), but 3 of 1000 8.6 against 8.2 (16)
    const int32_t max_chunks = force_split || total <= 64 ? 32 : 64;
    const int32_t short_cb = std::max(4, (int32_t)std::lround(0.25 * std::sqrt((double)total)));
    if (n > max_chunks) return total <= 64 ? 3 : short_cb;
    int32_t cb = fit(max_chunks);
    if (max_chunks == 64 && total <= 128 && n <= 32 && longest > 16 * cb) cb = fit(32);
    return cb - total / 64.0 <= 0.5 * std::sqrt((double)total) ? cb : short_cb;
}

}  // namespace kvc
