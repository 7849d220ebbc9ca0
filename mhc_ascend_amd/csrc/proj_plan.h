// Host-side rules of the projections that take only numbers: how a launch is
// split.  No HIP in here, so they run (and are tested) anywhere.
#pragma once
#include <stdint.h>

namespace mhc {

// ---- streaming projection (dynamic.hip) ---------------------------------------
struct StreamFill {
    int64_t groups;  // workgroups of one K split
    int64_t slots;   // resident workgroups
    int64_t stages;  // k stages
    int64_t kmax;    // most splits: two stages each, splits x tokens at most 4096
                     // (the partials the coefficient kernel adds per token)
};

inline StreamFill stream_fill_of(int64_t B, int64_t K, int np, int mt, int rows_per_wg, int k_per_stage,
                                 int64_t slots) {
    StreamFill f{};
    f.groups = (B + 16 * mt - 1) / (16 * mt) * ((np + rows_per_wg - 1) / rows_per_wg);
    f.slots = slots;
    f.stages = (K + k_per_stage - 1) / k_per_stage;
    const int64_t kcap = B > 0 ? (4096 + B - 1) / B : 1;
    f.kmax = (f.stages + 1) / 2 < kcap ? (f.stages + 1) / 2 : kcap;
    if (f.kmax < 1) f.kmax = 1;
    return f;
}

// Splits whose workgroups fill two rounds of the resident ones.
inline int64_t stream_fill_splits(const StreamFill& f) {
    int64_t ks = 2 * f.slots / f.groups;
    if (ks > f.kmax) ks = f.kmax;
    return ks < 1 ? 1 : ks;
}

// The count whose rounds of resident workgroups take the fewest stages, three
// added per workgroup for its prologue and stores; a larger count only where it
// takes 2% less.  n = 32, 128 tokens, C = 1280: 28 splits are 504 workgroups, one
// round; 32, the cap, left 64 of 576 to a second one (110 us, 88 with the
// workgroup order and the packed split of the kernel).
// (Of the counts with the same stages per split the first has the fewest rounds:
// the search steps from one to the next, some 2 sqrt(stages) of them.  It runs in
// every size query and launch; each count in turn took 1024 steps for a single
// token at n = 32, 4096 channels.)
inline int stream_ksplit(const StreamFill& f) {
    int64_t best = 1, best_cost = 0;
    for (int64_t ks = 1; ks <= f.kmax;) {
        const int64_t per = (f.stages + ks - 1) / ks;
        const int64_t cost = (f.groups * ks + f.slots - 1) / f.slots * (per + 3);
        if (ks == 1 || cost * 50 < best_cost * 49) {
            best = ks;
            best_cost = cost;
        }
        if (per <= 1) break;
        ks = (f.stages + per - 2) / (per - 1);
    }
    return (int)best;
}

}  // namespace mhc
