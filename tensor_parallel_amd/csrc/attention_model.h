// The cost model that cuts a decode step's keys into ranges (host code).
#pragma once
#include <math.h>
#include <stdint.h>

namespace tpamd {

constexpr int DECODE_MAX_SPLITS = 64;

// Key ranges per head of attention_decode_kernel: the count with the smallest predicted time (microseconds). A block alone reads its keys at 52 GB/s (head_dim 64: 40; it
// shares its CU with one other, four others for 64), all blocks together at 5.9 TB/s, 4 % less of it where they are more than the CUs: the busiest CU is then the last
// to end. Several ranges cost a second launch and their partials. Fitted to 722 timings in HIP graphs on caches that rotate through 2 GB (1 to 1024 heads on 16 to 131072 keys and 80
// random shapes, with a new position and without, each cut into 1 to 64 ranges): 0.4 % off the best count (geometric mean), at worst 8 %. Before, with 32 ranges at most and no cost beyond
// one block per CU, 2.0 % and 42 %: one head on 131072 keys 46 us in 32 ranges, 33 in 64; 16 heads on those 206 in 18 (288 blocks), 156 in 12; 96 heads on 2675 32 in 3, 25 in 2.
inline int decode_splits(int64_t heads, int64_t keys, int D, int cus) {
    constexpr int TILE = 64;  // ranges are whole tiles of this many keys
    double best = 1e30;
    int pick = 1;
    const int per_cu = D == 128 ? 2 : 5;
    const double alone = D == 128 ? 52.0e3 : 40.0e3, all = static_cast<double>(heads) * static_cast<double>(keys) * D * 4.0 / 5.9e6;
    for (int n = 1; n <= DECODE_MAX_SPLITS; ++n) {
        const int64_t kps = ((keys + n - 1) / n + TILE - 1) / TILE * TILE;
        if (n > 1 && (keys + kps - 1) / kps != n) continue;  // rounds to another count
        const double turns = static_cast<double>((heads * n + per_cu * cus - 1) / (per_cu * cus));
        const double own = turns * static_cast<double>(kps < keys ? kps : keys) * D * 4.0 / alone, together = heads * n > cus ? 1.04 * all : all;
        const double a2 = own * own, b2 = together * together;
        const double t = sqrt(sqrt(a2 * a2 + b2 * b2)) + (n > 1 ? 2.0 + 0.1 * n : 0.0);
        if (t < best) { best = t; pick = n; }
    }
    return pick;
}

}  // namespace tpamd
