// How the products that split K over the grid choose their splits: host arithmetic only (no HIP types), with the
// chip's compute units as a parameter, so that the same rules run in the launchers and in a CPU test of their
// invariants.  A split plan is what the launch, the kernel's indexing and the workspace query must agree on:
//   splits       blocks along the grid axis of K (1: no split, no workspace);
//   per_split    units of K per split, in the kernel's unit (steps of 64 values for the matrix-core kernels, rows of
//                the weight for the vector kernel); split i takes [i * per_split, min((i + 1) * per_split, units));
//   every split has at least one unit: (splits - 1) * per_split < units.
// The float32 partial sums are [batch][splits][m][n] (one batch for the tiled kernel of weights stored [N, K]).
#pragma once

#include <math.h>
#include <stddef.h>
#include <stdint.h>

#include <initializer_list>

#include "nuvec_hip.h"  // NVQ_STATIC_SCRATCH_BYTES

namespace nvq {
namespace splits {

// Microseconds a step of 64 values of K takes the tiled kernels of weights stored [N, K]: the 256 x 256 tile of qmm_kernel, qmk_kernel's
// tiles of 128 and of 64 rows, and qmm_kernel's 128 x 128 tile alone on a compute unit and where two of them share one.
struct StepTimes {
    float big, qmk128, qmk64, alone, shared;
};
// What the expansion of the codes decides: widths whose codes cross words (5 bits above all), two roundings a weight.
inline StepTimes step_times(int mode, int bits, bool float16, bool exact_weights) {
    if (mode == NVQ_MXFP4) return {1.05f, 0.36f, 0.273f, 0.456f, 0.67f};
    if (mode == NVQ_MXFP8) return {1.17f, 0.396f, 0.305f, 0.493f, 0.8f};
    if (mode == NVQ_NVFP4) return {1.45f, 0.43f, 0.37f, 0.714f, 0.97f};
    const int width = bits == 5 ? 2 : bits == 3 || bits == 6 ? 1 : 0;
    static constexpr StepTimes once[] = {{1.27f, 0.442f, 0.378f, 0.61f, 0.95f}, {1.32f, 0.49f, 0.44f, 0.71f, 1.07f}, {1.84f, 0.64f, 0.568f, 0.79f, 1.34f}};
    static constexpr StepTimes exact16[] = {{1.27f, 0.467f, 0.397f, 0.68f, 1.03f}, {1.32f, 0.524f, 0.476f, 0.766f, 1.16f}, {1.84f, 0.7f, 0.596f, 0.846f, 1.38f}};
    static constexpr StepTimes exact[] = {{1.27f, 0.533f, 0.469f, 0.91f, 1.36f}, {1.32f, 0.579f, 0.55f, 1.01f, 1.51f}, {1.84f, 0.74f, 0.66f, 1.085f, 1.76f}};
    return !exact_weights ? once[width] : float16 ? exact16[width] : exact[width];
}

struct Product {
    int64_t m, n, k, batch;
    bool row_exact;      // every row takes the split of its one-row product
    bool exact_weights;  // the tiled kernels of weights stored [N, K]: qmk_kernel's tiles
    StepTimes step = step_times(NVQ_AFFINE, 4, false, false);
};

struct Plan {
    int splits;
    int64_t per_split;  // units per split
    int64_t units;      // all units of K
    double estimate_us; // of the kernel with this plan, where the rule estimates one (else 0)
    int tile;           // tiled kernels of weights stored [N, K]: a Tile
};

inline bool every_split_has_a_unit(const Plan &p) {
    return p.splits >= 1 && p.per_split >= 1 && (int64_t)(p.splits - 1) * p.per_split < p.units &&
           (int64_t)p.splits * p.per_split >= p.units;
}
inline size_t workspace_bytes(const Plan &p, const Product &a) {
    return p.splits > 1 ? (size_t)p.splits * (size_t)a.batch * (size_t)a.m * (size_t)a.n * sizeof(float) : 0;
}

// ── the tiled kernels of weights stored [N, K] (qmm_kernel, qmk_kernel) ─────────────────────────────────────────────
constexpr int kQmmStep = 64;  // values of K per step; qmk_kernel takes two at a time
constexpr int kQmmBigTile = 256, kQmmSmallTile = 128, kQmkFewRows = 64;
enum Tile { kBig, kQmk128, kQmk64, kSmall };  // qmm_kernel's 256 x 256; qmk_kernel's 128 x 128 and 64 x 128; qmm_kernel's 128 x 128

inline int64_t qmm_tiles(const Product &a, int tile) {
    const int64_t rows = tile == kBig ? kQmmBigTile : tile == kQmk64 ? kQmkFewRows : kQmmSmallTile, cols = tile == kBig ? kQmmBigTile : kQmmSmallTile;
    return (a.m + rows - 1) / rows * ((a.n + cols - 1) / cols) * a.batch;
}
// The plan as it was made when qmm_kernel's 128 x 128 tile (0.8 us a step alone on a compute unit, 1.2 where two share it) stood where
// qmk_kernel's does: by whole tiles first, then the split of that tile.  What gated pairs and up to 32 rows were timed beside.
inline Plan qmm_plan_before(const Product &a, int cus) {
    const int64_t steps = (a.k + kQmmStep - 1) / kQmmStep;
    auto tiles_us = [&](int tile, double tiles, double each) {
        return tile == kBig ? ceil(tiles / cus) * each * 1.7 : tiles <= cus ? each * 0.8 : ceil(tiles / (2.0 * cus)) * each * 1.2;
    };
    const double big = tiles_us(kBig, (double)qmm_tiles(a, kBig), (double)steps), small = tiles_us(kQmk128, (double)qmm_tiles(a, kQmk128), (double)steps);
    const int tile = a.exact_weights || small < big ? kQmk128 : kBig;
    const double tiles = (double)qmm_tiles(a, tile), outputs = (double)a.m * (double)a.n;
    Plan p{1, steps, steps, tile == kBig ? big : small, tile};
    for (int want = 2; a.batch == 1 && want <= 8 && want <= steps / 8; want++) {
        const int64_t per = ((steps + want - 1) / want + 3) & ~(int64_t)3;
        const int splits = (int)((steps + per - 1) / per);  // every split has a step
        if (splits < 2 || (a.k % kQmmStep != 0 && (double)splits * outputs * 4.0 > (double)NVQ_STATIC_SCRATCH_BYTES)) continue;
        const double us = tiles_us(tile, tiles * splits, (double)per) + 3.0 + ((double)splits * 4.0 + 2.0) * outputs * 2.0 / 4.0e6;
        if (us < 0.9 * p.estimate_us) p.estimate_us = us, p.splits = splits, p.per_split = per;
    }
    return p;
}

// Estimated microseconds of `tiles` tiles walking `steps` steps each on `cus` compute units, in `splits` parts of K whose sums a second
// kernel adds up: a launch, for each round of tiles its first loads and its end, the steps (longer by what the compute units share where
// all are busy), the outputs.  Fitted (least squares of the relative error, 5 to 7 % off by kernel) to 19000 timings of 1980 products: 17 to
// 2048 rows, W[256..40000, 64..32768], all formats of 16-bit elements, one to eight parts.
inline float qmm_tiles_us(const Product &a, int tile, int64_t tiles, int64_t steps, int splits, int cus) {
    const float outputs = 1.0e-6f * (float)(a.m * a.n * a.batch), parts = splits > 1 ? splits * outputs : 0.0f, each = (float)steps;
    const float rounds = (float)((tiles + cus - 1) / cus), busy = (float)tiles / (float)cus * each, two = splits > 1 ? 1.0f : 0.0f;
    switch (tile) {
    case kBig: return 10.9f + rounds * (2.6f + a.step.big * each) + 0.337f * busy + 1.02f * parts;
    case kQmk128: return 4.2f + rounds * (2.34f + a.step.qmk128 * each) + 0.081f * busy + 0.63f * outputs + 2.2f * two + 1.36f * parts;
    case kQmk64: return 2.6f + rounds * (1.9f + a.step.qmk64 * each) + 0.034f * busy + 0.65f * outputs + 2.8f * two + 1.13f * parts;
    default: return 5.4f + (tiles <= cus ? a.step.alone : (float)((tiles + 2 * cus - 1) / (2 * cus)) * a.step.shared) * each + 0.096f * busy + 0.25f * outputs;
    }
}

// The tile and the split of K with the least estimated time (1980 products of 17 to 2048 rows by it and the other kernels' estimates: 0.87 of
// the time before qmk_kernel, one in 60 more than 5 % slower, where one in 30 differs by that between two runs of one side).  The splits fill the compute units with few tiles.  Each split has at least
// eight steps, in whole windows and table periods (four steps); at most eight splits; a batch is never split.  K is split as far as the
// library's own scratch holds the partial sums, so that the entry point without a workspace refuses no product that it took: all up to
// K = 14336 and of steps and a half, longer ones whose former plan fitted or that other kernels may have taken.  (Beyond the scratch five splits are no faster than two: 768 rows,
// W[8192,32768] of 4 bits 395 and 395 us.)
inline Plan qmm_plan(const Product &a, int cus) {
    if (cus < 1) cus = 1;
    const int64_t steps = (a.k + kQmmStep - 1) / kQmmStep;  // (the last one may be a half)
    const bool capped = a.k <= 14336 || a.k % kQmmStep != 0 || a.m <= 640 || a.exact_weights || workspace_bytes(qmm_plan_before(a, cus), a) <= (size_t)NVQ_STATIC_SCRATCH_BYTES;
    Plan best{0, 0, 0, 0.0, 0};
    for (const int tile : {kBig, kQmk128, kQmk64, kSmall}) {
        const int64_t tiles = qmm_tiles(a, tile), high = (a.m + (tile == kQmk64 ? kQmkFewRows : kQmmSmallTile) - 1) / (tile == kQmk64 ? kQmkFewRows : kQmmSmallTile);
        if (tile == kBig && a.exact_weights) continue;
        if (tile != kBig && high > 65535 && !(a.exact_weights && tile == kQmk128)) continue;  // (the grid's rows)
        if (tile == kSmall && a.exact_weights && (a.batch != 1 || a.k % kQmmStep != 0)) continue;  // (has single products of whole steps)
        Plan p{1, steps, steps, qmm_tiles_us(a, tile, tiles, steps, 1, cus), tile};
        const int64_t most = a.batch == 1 && tiles < 2 * cus && tile != kSmall ? (steps < 64 ? steps / 8 : 8) : 1;  // (more tiles fill the chip as they are)
        for (int want = 2; want <= most; want++) {
            const int64_t per = ((steps + want - 1) / want + 3) & ~(int64_t)3;
            const int splits = (int)((steps + per - 1) / per);  // every split has a step
            if (splits < 2) continue;
            if (capped && (double)splits * (double)a.m * (double)a.n * 4.0 > (double)NVQ_STATIC_SCRATCH_BYTES) break;
            const float us = qmm_tiles_us(a, tile, tiles * splits, per, splits, cus);
            if (us < 0.97f * (float)p.estimate_us) p.estimate_us = us, p.splits = splits, p.per_split = per;
            if (tiles * splits >= 2 * cus) break;
        }
        if (best.splits == 0 || p.estimate_us < best.estimate_us) best = p;
    }
    return best;
}

// What the kernels of a tiled plan take for granted; NULL where it holds, else what does not.  A split reads its tables from a period's start
// and qmk_kernel walks whole windows of two steps; of the weights with two roundings qmm_kernel has the 128 x 128 tile of whole steps alone.
inline const char *qmm_plan_fault(const Plan &p, const Product &a) {
    if (p.units != (a.k + kQmmStep - 1) / kQmmStep || !every_split_has_a_unit(p)) return "a part of K without a step";
    if (p.splits > 1 && a.batch != 1) return "a batch whose K is split";
    if (p.splits > 1 && p.per_split % 4 != 0) return "parts of K that are no whole table periods";
    if (a.exact_weights && (p.tile == kBig || (p.tile == kSmall && (a.batch != 1 || a.k % kQmmStep != 0)))) return "a tile that does not round these weights twice";
    return nullptr;
}

// ── the matrix-core kernel of weights stored [K, N] (qmn_kernel) ────────────────────────────────────────────────────
constexpr int kQmnStep = 64, kQmnTileCols = 128;
constexpr int kQmnFewRows = 32, kQmnManyRows = 128;          // rows of x per tile
constexpr int kQmnFewBlocksPerCu = 4, kQmnManyBlocksPerCu = 2;

// Splits of K for a product whose tiles do not fill the chip: the split with the least estimated time, counted as
// rounds of resident blocks x (3 us to start + 1.2 us per step of the longest split; 0.64 us per step of the 32-row
// tile) plus, with a split, the reduction: its launch, 0.38 us per split it adds up in turn and its float32 traffic at
// 4 TB/s (fitted to w[4096,4096] at 1 to 32 rows: 43 / 26 / 17 / 13 / 15 / 20 us with 1 / 2 / 4 / 8 / 16 / 32 splits).
inline Plan qmn_plan(const Product &a, int cus, bool few_rows) {
    const int64_t bm = few_rows ? kQmnFewRows : kQmnManyRows;
    const int64_t tiles = ((a.m + bm - 1) / bm) * ((a.n + kQmnTileCols - 1) / kQmnTileCols) * a.batch, steps = a.k / kQmnStep;
    const int64_t resident = (int64_t)(few_rows ? kQmnFewBlocksPerCu : kQmnManyBlocksPerCu) * cus;
    Plan p{1, steps < 1 ? 1 : steps, steps, 0.0, 0};
    if (tiles >= resident || steps < 4) return p;
    const double step_us = few_rows ? 0.64 : 1.2;
    for (int64_t splits = 1; splits <= steps / 2 && splits <= 64; splits++) {
        const int64_t per_split = (steps + splits - 1) / splits;
        if ((steps + per_split - 1) / per_split != splits) continue;  // (another count gives the same longest split)
        const int64_t rounds = (tiles * splits + resident - 1) / resident;
        double us = (double)rounds * (3.0 + step_us * (double)per_split);
        if (splits > 1) us += 2.0 + 0.38 * (double)splits + (double)splits * (double)(a.batch * a.m * a.n) * 4.0 / 4.0e6;
        if (splits == 1 || us < p.estimate_us) p.estimate_us = us, p.splits = (int)splits, p.per_split = per_split;
    }
    return p;
}

// ── the vector kernel of weights stored [K, N] (qvm_kernel) ─────────────────────────────────────────────────────────
constexpr int kQvmWaves = 8, kQvmTileCols = 2048;

// About a block (of eight wavefronts) per compute unit, at least 16 rows of w per wavefront, at most 32 splits (the
// reduction kernel adds them one after the other).  The unit is a row of the weight.
inline Plan qvm_plan(const Product &a, int cus) {
    const int rm = a.m == 1 ? 1 : 4;
    // row-exact: the split is the one-row product's, whatever the rows and batches, so that every row keeps its bits
    const int64_t base = ((a.n + kQvmTileCols - 1) / kQvmTileCols) * (a.row_exact ? 1 : a.batch * ((a.m + rm - 1) / rm));
    const int64_t want = ((int64_t)cus + base - 1) / base;
    const int64_t most = a.k / (16 * kQvmWaves) > 1 ? a.k / (16 * kQvmWaves) : 1;
    int64_t splits = want < 1 ? 1 : (want > most ? most : want);
    if (splits > 32) splits = 32;
    int64_t per = (a.k + splits - 1) / splits;
    if (per < 1) per = 1;
    splits = (a.k + per - 1) / per;  // the count that this longest split gives: no split is left without a row
    if (splits < 1) splits = 1;
    return Plan{(int)splits, per, a.k, 0.0, 0};
}

}  // namespace splits
}  // namespace nvq
