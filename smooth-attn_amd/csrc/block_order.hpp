// Host-side choice of the attention grids' block order: how many units
// (KV heads) an XCD takes at a time (grouped_block in flash_common.hpp).
#pragma once

#include <algorithm>
#include <cstdint>
#include <functional>
#include <vector>

namespace sa {

// Units per group: the fewest whose blocks fill an XCD's slots, or, where
// steps differ in work (`uneven`), all of the XCD's as one group.
//
// Where a group's blocks are no multiple of xcd_slots, the next group's heavy
// steps start late and the last group's end late, up to half again the
// balanced time in grids of a few rounds.  Up to kOneGroupRounds blocks per
// slot an XCD then takes all its units as one group, heavy steps first
// throughout.  Longer grids lose more L2 hits than they gain ([4,32,5000], 10
// rounds, forward / backward 931 / 3022 -> 934 / 3080 us).
//
// One group's time over groups', in geometric mean and at worst, over random
// shapes (T = 300 to 8192) that take it: forward at D <= 64 (37 shapes) 0.93
// and 1.03, at D = 80 to 128 see order_gain; backward, windows included, (130)
// 0.92 and 1.04 ([6,64/8,319,96] 97 -> 101 us); forward at D = 136 to 512,
// windows included, (8 of 60 differ) 0.72 to 0.99.  [1,32,3000,128] 126 / 397 ->
// 102 / 341 us, [2,32,1536,128] 71 / 227 -> 58 / 193, [1,32,1344,256] forward
// 57 -> 46.
constexpr int kOneGroupRounds = 8;
inline int units_per_group(int n_units, int n_sub, int n_steps, int xcd_slots, bool uneven) {
    // blocks of a unit (none in an empty call, which launches nothing), units of an XCD
    const int per = n_sub * n_steps > 0 ? n_sub * n_steps : 1, units = n_units >> 3;
    int gu = (xcd_slots + per - 1) / per;
    if (gu < 1) gu = 1;
    if (gu > units) gu = units;
    if (uneven && units * per <= kOneGroupRounds * xcd_slots && gu * per % xcd_slots != 0) gu = units;
    return gu;
}

// Time of one XCD's blocks in groups of gu units, each block starting on the
// slot that frees first; cost(step): a block's.
template <typename Cost>
double order_makespan(int units, int n_sub, int n_steps, int gu, int xcd_slots, Cost cost) {
    std::vector<double> slots(static_cast<size_t>(xcd_slots), 0.0);
    for (int u0 = 0; u0 < units; u0 += gu) {
        const int heads = std::min(gu, units - u0) * n_sub;
        for (int step = 0; step < n_steps; ++step) {
            const double c = cost(step);
            for (int i = 0; i < heads; ++i) {
                std::pop_heap(slots.begin(), slots.end(), std::greater<double>());
                slots.back() += c;
                std::push_heap(slots.begin(), slots.end(), std::greater<double>());
            }
        }
    }
    return *std::max_element(slots.begin(), slots.end());
}

// Whether one group shortens the time by enough to pay for its L2 hits.  For
// the forward at D = 80 to 128 (one block per CU) the estimate separates 73
// random shapes: from 6% on one group takes 0.90 of the groups' time, at worst
// 1.04, below it 1.02 and up to 1.06 ([3,32,1359,128] 70.5 -> 75.2 us).  At D <=
// 64 (two blocks per CU) and in the backward one group wins below it, too.
// About 10 us of host time.
constexpr double kOneGroupGain = 1.06;
template <typename Cost>
bool order_gain(int n_units, int n_sub, int n_steps, int gu, int xcd_slots, Cost cost) {
    const int units = n_units >> 3;
    return order_makespan(units, n_sub, n_steps, gu, xcd_slots, cost) >=
           kOneGroupGain * order_makespan(units, n_sub, n_steps, units, xcd_slots, cost);
}

}  // namespace sa
