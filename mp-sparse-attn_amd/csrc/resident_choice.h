// When many queries over few keys go to the kernel that keeps a head's K and V in LDS (attn_fwd_resident.hip) instead of the one
// that streams them (attn_fwd_short.hip, one split), and how its work is shared out.  No HIP in here: the host compiler builds it for
// its test.
#pragma once
#include <stdint.h>

constexpr int RESIDENT_WAVES = 8;

// Workgroups that share a (batch, KV head) of `tasks` blocks of 32 queries, 256 at most: the fewest clocks of rounds of 256 workgroups,
// each the way into LDS of nb blocks of 32 keys and its waves' blocks.  Of the numbers with which a wave has the same number of blocks
// the least is the best; the others are passed over (1000 times eight blocks: 60 numbers looked at instead of 256).
inline int64_t resident_shares(int64_t units, int64_t tasks, int64_t nb) {
    const int64_t eights = (tasks + RESIDENT_WAVES - 1) / RESIDENT_WAVES;
    int64_t best = INT64_MAX, shares = 1;
    for (int64_t x = 1; x <= eights && x <= 256;) {
        const int64_t waves = (eights + x - 1) / x, clocks = (units * x + 255) / 256 * (13000 + 250 * nb + waves * (6800 + 1000 * nb));
        if (clocks < best) {
            best = clocks;
            shares = x;
        }
        if (waves == 1) break;
        x = (eights - 1) / (waves - 1) + 1;
    }
    return shares;
}

// The workgroups per (batch, KV head), or 0 where the streaming kernel is estimated to be the faster one.  Microseconds of either,
// fitted to measurements at 9000 shapes (1 to 2048 heads, 1 to 32768 queries, 8 to 448 keys, 8-bit and mixed): a round of 256 workgroups
// costs the way into LDS and as many blocks of queries as its longest wave has; the streaming kernel's workgroups of 128 queries, two a
// CU, cost more by their number; and either by the queries it moves.  Over the 8600 of these shapes that the choice of kernels
// brings here it costs 0.5 % over always taking the faster one, where taking every call from 4096 blocks of 32 queries on cost 3.6 %:
// up to 1.48 times the time where a head has few queries (64 x 16 heads of 128 over 333 keys 46.5 us streamed, 67.8 here),
// and 1.07 to 1.10 over 32 keys or fewer however many queries there are.  From 3072 blocks on: below, the two are within 2 % of each
// other in the mean and the estimates no longer tell them apart.
inline int64_t resident_choice(int64_t B, int64_t Hq, int64_t Hkv, int64_t nq, int64_t nk) {
    const int64_t blocks = B * Hq * ((nq + 31) / 32);
    if (blocks < 3072) return 0;
    const int64_t units = B * Hkv, tasks = Hq / Hkv * ((nq + 31) / 32), nb = (nk + 31) / 32;
    const int64_t shares = resident_shares(units, tasks, nb);
    const double rounds = (double)((units * shares + 255) / 256), waves = (double)((tasks + RESIDENT_WAVES * shares - 1) / (RESIDENT_WAVES * shares));
    const double here = 3.5 + rounds * (0.589 + 0.436 * nb + waves * (3.031 + 0.387 * nb)) + 1.965e-3 * blocks;
    const int64_t workgroups = B * Hq * ((nq + 127) / 128);
    double load = workgroups / 512.0;
    load = 0.481 * (load > 1.0 ? load : 1.0) + 0.519 * ((workgroups + 511) / 512);
    const double streamed = 5.7 + load * (2.402 + 0.722 * nb) + 1.901e-3 * blocks;
    return here < streamed ? shares : 0;
}
