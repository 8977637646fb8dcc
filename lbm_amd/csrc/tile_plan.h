// How a call of many steps is cut into launches of several steps each (tile.h,
// lbm_f64.hip): the block shapes, what a launch costs, and the choice.  Host
// code but for the region counts, which the kernels share; no HIP calls, so that
// it also builds into plain C++ checks.
#pragma once

#include <algorithm>
#include <cmath>
#include <cstdint>

#include "../../include/lbm_hip.h"

namespace {

constexpr int kTileMaxSteps = 8;
// steps an autotuner times a tile variant for at least: launches of a few steps
// (two of three in a call of six) say little about those of a long call
constexpr uint32_t kTileTimedSteps = 48;
// A tuning call of fewer steps does not time the tile variants (it asks for the
// fastest single step); then neither do its results turn the default path off.
constexpr uint32_t kTileTunedFrom = 3;

// Block shapes of k_tile: rows a wave, waves, where the unstreamed cells' previous
// populations live, and the launch's cost.  Without `chain` every cell has a
// place for them in LDS and solid cells are stepped like any other; with it only
// column 0, column X and the last row have one and solid cells, which nothing
// pulls from, are stepped on their own at the end (three rows a wave would need
// 72 KB a block more).
//
// us = fixed + step * steps + rounds * (block + block_step * steps), rounds the
// regions each CU works off one after the other: fitted to launches of 2 to 8
// steps over 0.06 to 33 million cells (within 9% / 32% / 14% / 16%, the largest
// errors where a round is barely begun).
struct TileShape {
    int m, waves;
    bool chain;
    float fixed, step, block, block_step;
};
constexpr TileShape kTileF32[2] = {{1, 16, false, 2.18f, 0.58f, 2.43f, 0.26f}, {3, 12, true, 0.0f, 2.28f, 7.6f, 0.53f}};
constexpr TileShape kTileF16[2] = {{1, 16, false, 2.28f, 0.56f, 2.33f, 0.29f}, {2, 16, false, 1.7f, 1.03f, 4.73f, 0.6f}};
template <class T>
constexpr const TileShape &tile_shape(int i) { return sizeof(T) == 4 ? kTileF32[i] : kTileF16[i]; }
inline const TileShape &tile_shape(int precision, int i) {
    return precision == LBM_PRECISION_F32 ? kTileF32[i] : kTileF16[i];
}

// regions that cover n cells when each of `size` cells keeps all but 2 h
constexpr int tile_regions(int n, int size, int h) {
    return n <= size ? 1 : 1 + (n - size + (size - 2 * h) - 1) / (size - 2 * h);
}
// (column X counts: the outlet's wrapped pulls; so does the row above the grid)
constexpr int tile_nbx(int X, int steps) { return tile_regions(X + 1, 64, steps - 1); }
constexpr int tile_nby(int Y, int rows, int steps) { return tile_regions(Y + 1, rows, steps - 1); }

inline float tile_cost(const TileShape &sh, int steps, double blocks) {
    double rounds = std::max(1.0, blocks / 256.0);
    if (rounds < 4.0) rounds = std::ceil(rounds);
    return (float)(sh.fixed + sh.step * steps + rounds * (sh.block + sh.block_step * steps));
}

// the fewest launches of up to s steps that make n (n + s - 1 may not fit)
inline uint32_t launches_of(uint32_t n, int s) { return n / (uint32_t)s + (n % (uint32_t)s != 0); }

// How a call of n >= 2 steps is cut into launches, each of them n / launches
// steps or one more: the shape (of `first` .. `last`) and number of launches of
// least cost (no launches: none fits a grid of blocks).  blocks(shape index,
// steps): the regions of a launch.
struct TilePlan {
    int shape;
    uint32_t launches;
};
//
// even: an even number of launches, whatever n is (none for calls of two or three
// steps).  Every launch trades the state and spare sets; after an even number
// each is where it was, as after the one-step kernel's calls.  A caller's graph
// of a call holds the sets it was captured with, and needs that of every call.
template <class F>
TilePlan tile_plan(int precision, int first, int last, uint32_t n, bool even, F &&blocks) {
    TilePlan best{first, 0};
    float least = 0.0f;
    for (int i = first; i <= last; ++i) {
        const TileShape &sh = tile_shape(precision, i);
        float cost[kTileMaxSteps + 1] = {};
        for (int s = 2; s <= kTileMaxSteps; ++s) {
            const int64_t nb = blocks(i, s);
            cost[s] = nb * 64 * sh.waves < (int64_t)1 << 32 ? tile_cost(sh, s, (double)nb) : INFINITY;
        }
        for (int s = 2; s <= kTileMaxSteps; ++s) {
            uint32_t launches = launches_of(n, s);
            if (even) launches += launches % 2;
            const uint32_t low = n / launches;
            if (low < 2) continue;
            const uint32_t more = n % launches;
            const float c = cost[low] * (float)(launches - more) + (more ? cost[low + 1] * (float)more : 0.0f);
            if (std::isfinite(c) && (!best.launches || c < least)) {
                best = TilePlan{i, launches};
                least = c;
            }
        }
    }
    return best;
}

// Block shapes of the FP64 solver's k64_tile (lbm_f64.hip), the cost fitted to
// launches of 1 to 8 steps over 0.006 to 4 million cells (within 20% / 38% / 44%,
// the largest errors where a round is barely begun).  Best us per step of each: 300 x 150 1.95 / 2.71 / 3.88, 640 x
// 320 4.24 / 3.65 / 4.05, 2048 x 1024 32.4 / 22.7 / 20.2.  Taller regions of
// three and four rows a wave leave one block a CU, whose loads nothing then
// hides (3 x 12: 25.9, 4 x 12: 25.7).
constexpr TileShape kTile64[3] = {{1, 16, false, 0.0f, 0.37f, 5.47f, 0.66f},
                                  {2, 12, false, 0.0f, 0.93f, 6.67f, 0.95f},
                                  {4, 8, false, 0.0f, 1.17f, 8.21f, 1.48f}};

// A call's launches: their number is odd, as they go from g to f to g ... and
// the last one has to end in f, which holds the cells the stream does not write.
inline TilePlan plan64(int X, int Y, uint32_t n) {
    TilePlan best{0, 0};
    float least = 0.0f;
    for (int i = 0; i < 3; ++i) {
        const TileShape &sh = kTile64[i];
        float cost[kTileMaxSteps + 2] = {};
        for (int s = 1; s <= kTileMaxSteps; ++s)
            cost[s] = tile_cost(sh, s, (double)tile_nbx(X, s) * tile_nby(Y, sh.waves * sh.m, s));
        for (int s = 1; s <= kTileMaxSteps; ++s) {
            const uint32_t launches = launches_of(n, s) | 1u;
            if (launches > n) continue;
            const uint32_t low = n / launches, more = n % launches;
            const float c = cost[low] * (float)(launches - more) + cost[low + 1] * (float)more;
            if (!best.launches || c < least) {
                best = TilePlan{i, launches};
                least = c;
            }
        }
    }
    return best;
}

}  // namespace
