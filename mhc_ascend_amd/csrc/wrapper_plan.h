// Host-side rules of the wrapper's kernels that take only numbers: how a
// launch is split.  No HIP in here, so they run (and are tested) anywhere.
#pragma once
#include <stdint.h>

namespace mhc {

// ---- folded forward projection (wrapper_proj.hip) ----------------------------
// Waves per workgroup: eight at 64 tokens a wave of bf16 rows, so that two
// waves of a SIMD overlap one's residual arithmetic with the other's MFMAs while
// Phi still crosses LDS once per 512 tokens; four otherwise (fp32 rows' split
// operands need more than 256 registers).
constexpr int wp_waves(int dt_size, int tw) { return dt_size == 2 && tw == 4 ? 8 : 4; }

// 16-row tiles of a row block: all of them up to six, else the count that
// pads least (the larger on ties: fewer passes over the rows).
inline int wfold_rt(int np) {
    const int tiles = (np + 15) / 16;
    if (tiles <= 6) return tiles;
    int best = 6;
    for (int rt = 5; rt >= 4; --rt) {
        if ((tiles + rt - 1) / rt * rt * (rt + 1) * best < (tiles + best - 1) / best * best * (best + 1) * rt) best = rt;
    }
    return best;
}

inline int wfold_row_blocks(int np) {
    const int rt = wfold_rt(np);
    return ((np + 15) / 16 + rt - 1) / rt;
}

// Token tiles per wave: four (512 tokens a workgroup) where that still leaves
// enough workgroups, fewer for few tokens (a workgroup's rows past the batch
// are wasted, and every workgroup reads all of its Phi steps).
inline int wfold_tw(int64_t B) { return B >= 2048 ? 4 : (B >= 512 ? 2 : 1); }
inline int64_t wfold_tokens(bool bf16, int64_t B) {
    const int tw = wfold_tw(B);
    return (int64_t)16 * tw * wp_waves(bf16 ? 2 : 4, tw);
}

// Steps of 32 channels; bf16 rows take them in pairs (64 channels).
inline int wfold_steps(bool bf16, int64_t C) {
    return bf16 ? 2 * (int)((C + 63) / 64) : (int)((C + 31) / 32);
}

// Channel splits: one workgroup per CU, at least four steps a split, every
// split with a first step of its own (ks counts whole runs of `chunk` steps, so
// (ks - 1) chunk < steps: a run past the last step would read past the packed
// Phi, and its partials would be added for nothing).
struct WfoldSplit {
    int ks, chunk, steps;
};

inline WfoldSplit wfold_split(bool bf16, int64_t B, int64_t C, int np, int cus) {
    WfoldSplit s{};
    s.steps = wfold_steps(bf16, C);
    const int64_t per = wfold_tokens(bf16, B);
    const int64_t blocks = (B + per - 1) / per * wfold_row_blocks(np);
    int64_t ks = cus / (blocks < 1 ? 1 : blocks);
    if (ks > s.steps / 4) ks = s.steps / 4;
    if (ks < 1) ks = 1;
    s.chunk = (int)((s.steps + ks - 1) / ks);
    if (bf16) s.chunk = (s.chunk + 1) / 2 * 2;
    s.ks = (s.steps + s.chunk - 1) / s.chunk;
    return s;
}

// ---- dynamic-H backward (wrapper_bwd.hip) --------------------------------------
constexpr int kWbwdCols = 128;   // channels per workgroup
constexpr int kWbwdRound = 96;   // tokens of a round of its pipeline (three stages)

// Rows of a tile: each buffer (4 C bytes a row at most, or dP's row) under 2 GiB
// with the pipeline's overrun of six stages.
inline int64_t wbwd_max_tile(int64_t C, int64_t dp_row) {
    return ((int64_t(1) << 31) - 1) / ((C > dp_row ? C : dp_row) * 4) - 6 * 32;
}

// Tokens of each of `tiles` tiles.
inline int64_t wbwd_tile(int64_t B, int64_t tiles) {
    return ((B + tiles - 1) / tiles + kWbwdRound - 1) / kWbwdRound * kWbwdRound;
}

// Token tiles: one workgroup fits a CU (250 VGPRs, 8 waves), so column blocks x
// tiles is one to four rounds of workgroups, whichever leaves the fewest CUs
// idle in the last one (at 56 column blocks one round has 224 workgroups and
// took 1.42 ms at n = 8, two have 504 and took 1.28); whole pipeline rounds each
// and none without tokens, at most wbwd_max_tile (which holds one round at least).
inline int64_t wbwd_split(int64_t B, int64_t C, int64_t dp_row, int64_t cus) {
    const int64_t gx = (C + kWbwdCols - 1) / kWbwdCols;
    int64_t tiles = 1, best = 0;
    for (int64_t k = 1; k <= 4; ++k) {
        const int64_t fill = k * cus / gx * gx * 1000 / (k * cus);
        if (fill > best + 20) {
            best = fill;
            tiles = k * cus / gx;
        }
    }
    const int64_t rounds = (B + kWbwdRound - 1) / kWbwdRound;
    if (tiles > rounds) tiles = rounds;
    if (tiles < 1) tiles = 1;
    const int64_t mt = wbwd_max_tile(C, dp_row) / kWbwdRound * kWbwdRound;
    if (mt >= kWbwdRound && wbwd_tile(B, tiles) > mt) tiles = (B + mt - 1) / mt;
    const int64_t tile = wbwd_tile(B, tiles);
    return tile > 0 ? (B + tile - 1) / tile : 1;
}

}  // namespace mhc
