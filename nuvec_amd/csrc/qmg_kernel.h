// The grouped (sorted) gathered product of mixture-of-experts layers on the gfx950 matrix cores: the rows of x that belong to expert e,
// [offsets[e], offsets[e+1]), times that expert's weights, every weight decoded once per pass of 64 rows.  Counterpart of the reference's
// `gather_qmm_rhs` (crates/nuvec-kernels/src/metal/quantized.h:3301-3449, schedule at 2866-2906); values follow nuvec's CPU product
// (crates/nuvec-core/src/quantized.rs:679-719, crates/nuvec-core/src/kernels.rs:1091-1142) within the stated tolerance.  Affine weights
// are rounded once to the element type as in qmf_kernel.h, the CPU's, or float32 in terms (weights_in_terms).  The rows of one plain
// product may be the one group.
//
// A block owns 128 weight rows of one expert and a pass of up to 64 of its rows of x; its groups of four wavefronts run the loop of
// rows_body.h over a part of K each, and their sums meet in LDS.  The pass has one to four tiles of 16 rows, each number an
// instantiation of the loop: a pass of a few rows neither brings nor multiplies the others.  Gate and up rows that alternate in runs
// of 64 are the two tiles of one wavefront, lane for lane, so that the gated activation needs no exchange.
//
// What bounds it: the way of codes and x through a compute unit's memory pipeline, and the blocks' first loads (30 rows of each of 32
// experts, MXFP4 w[5760,2880], 91 us: 88 without the arithmetic, 77 without x as well, the arithmetic on operands that are not loaded 50).  Four blocks a compute unit with the loads of four windows under way; codes staged in LDS with x took the
// same time at two blocks, wider blocks of eight wavefronts (half the reads of x) 109 us against 97, codes read by lines of 128 bytes
// the same.  Before -> now (the kernel of four wavefronts on 32 x 32 x 16 tiles), us: that product at 8 / 30 / 40 rows an expert 90 / 105 / 124
// -> 82 / 95 / 108; 4 bits 130 / 134 / 163 -> 107 / 119 / 131; 8 bits 250 / 258 / 274 -> 142 / 156 / 168; w[768,2432] of 8 bits, 12 rows, 46 -> 21.
#pragma once

#include "rows_body.h"

namespace nvq {
namespace qmg {

using rows::kTile;
constexpr int kThreads = 64 * rows::kWaves;  // of a group, which shares x; the groups of a block split K
constexpr int kRows = 128;     // weight rows of a block: two tiles a wavefront, 64 rows apart
constexpr int kPassRows = 64;  // rows of x of a pass, the most
constexpr int most_groups(int hold) { return hold == rows::kTerms ? 2 : 4; }  // (weights in terms take more registers)
constexpr int stages(int mt, int bits, int hold) { return mt > 2 ? 2 : bits <= 4 && hold != rows::kTerms ? 4 : 3; }

template <typename T, int BITS, int FP4, int HOLD, int MT>
__device__ __forceinline__ void run_pass(const ProductArgs &a, unsigned char *lds, int e, int pass, int rows, int n0) {
    using B = rows::Body<T, BITS, FP4, HOLD, MT, 2, stages(MT, BITS, HOLD)>;
    const int tid = threadIdx.x & (kThreads - 1), lane = tid & 63, l = lane & 15, q = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), group = __builtin_amdgcn_readfirstlane(threadIdx.x / kThreads);
    const int groups = __builtin_amdgcn_readfirstlane(blockDim.x / kThreads);
    const int K = (int)a.k, N = (int)a.n;
    const int turns = ((K + rows::kWin - 1) / rows::kWin + groups - 1) / groups, k0 = group * turns * rows::kWin;
    floatx4_t acc[MT][2];
#pragma unroll
    for (int m = 0; m < MT; m++)
#pragma unroll
        for (int t = 0; t < 2; t++) acc[m][t] = floatx4_t{0.0f, 0.0f, 0.0f, 0.0f};
    auto xrow = [&](int r) {  // an index beyond x is the caller's error: clamped
        const int at = pass + (r < rows ? r : rows - 1);
        return a.lhs != nullptr ? min((int64_t)a.lhs[at], a.x_batches - 1) : (int64_t)at;
    };
    auto weight_row = [&](int t, int r) {
        const int n = n0 + 64 * t + kTile * wave + r;
        return n < N ? n : N - 1;  // (tail rows are not stored)
    };
    const int k1 = min(k0 + turns * rows::kWin, K);
    B::run(a, lds + group * B::kLdsBytes, wave, e, n0, k0, k1, turns, xrow, weight_row, acc);
    if constexpr (HOLD == rows::kTerms) rows::sum_plainly<T, BITS, MT, 2>(a, e, k0, k1, xrow, weight_row, acc);
    if (groups > 1) {  // the groups' sums, added in order by the first group's threads
        float *part = reinterpret_cast<float *>(lds);
        __syncthreads();
        if (group > 0) {
#pragma unroll
            for (int m = 0; m < MT; m++)
#pragma unroll
                for (int t = 0; t < 2; t++)
#pragma unroll
                    for (int i = 0; i < 4; i++) part[((group - 1) * MT * 8 + (m * 2 + t) * 4 + i) * kThreads + tid] = acc[m][t][i];
        }
        __syncthreads();
        if (group > 0) return;
        for (int g = 0; g < groups - 1; g++)
#pragma unroll
            for (int m = 0; m < MT; m++)
#pragma unroll
                for (int t = 0; t < 2; t++)
#pragma unroll
                    for (int i = 0; i < 4; i++) acc[m][t][i] += part[(g * MT * 8 + (m * 2 + t) * 4 + i) * kThreads + tid];
    }

    // Element i of lane (q, l): weight row 4 q + i of the tile, row l of x.
    const bool vector = N % 8 == 0;  // (four outputs of a lane are one store)
    const int col0 = n0 + kTile * wave + 4 * q;
    float bias[2][4];
    if (a.expert_bias != nullptr) {
        const T *from = (const T *)a.expert_bias + (int64_t)e * N;
#pragma unroll
        for (int t = 0; t < 2; t++)
#pragma unroll
            for (int i = 0; i < 4; i++) bias[t][i] = Elem<T>::load(from, col0 + 64 * t + i < N ? col0 + 64 * t + i : N - 1);
    }
    uint32_t places[MT];
#pragma unroll
    for (int m = 0; m < MT; m++) {
        const int r = pass + min(kTile * m + l, rows - 1);
        places[m] = a.out_rows != nullptr ? (uint32_t)min((int64_t)a.out_rows[r], a.batch - 1) : (uint32_t)r;
    }
    T *y = (T *)a.y;
    auto store = [&](int64_t at, int room, const float (&o)[4]) {
        if (vector) {
            if (room > 0) *reinterpret_cast<uint2 *>(y + at) = make_uint2(qmf::Ops<T>::pack(o[0], o[1]), qmf::Ops<T>::pack(o[2], o[3]));
        } else {
#pragma unroll
            for (int i = 0; i < 4; i++)
                if (i < room) Elem<T>::store(y, at + i, o[i]);
        }
    };
#pragma unroll
    for (int m = 0; m < MT; m++) {
        if (kTile * m + l >= rows) continue;
        float v[2][4];
#pragma unroll
        for (int t = 0; t < 2; t++)
#pragma unroll
            for (int i = 0; i < 4; i++)  // the expert's bias: added to the product as its output holds it, a separate rounded addition
                v[t][i] = a.expert_bias != nullptr ? Elem<T>::add(rounded<T>(acc[m][t][i]), bias[t][i]) : acc[m][t][i];
        if (a.glu != 0) {  // (N is whole runs of 128)
            const int hcol = (n0 >> 1) + kTile * wave + 4 * q;
            float o[4];
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const float g = rounded<T>(v[0][i]), up = rounded<T>(v[1][i]);
                o[i] = a.glu == 1 + NVQ_GLU_SWIGLU       ? glu<T, NVQ_GLU_SWIGLU>(g, up, a.glu_alpha, a.glu_limit)
                       : a.glu == 1 + NVQ_GLU_SWIGLU_OAI ? glu<T, NVQ_GLU_SWIGLU_OAI>(g, up, a.glu_alpha, a.glu_limit)
                                                         : glu<T, NVQ_GLU_GEGLU>(g, up, a.glu_alpha, a.glu_limit);
            }
            store((int64_t)places[m] * (N >> 1) + hcol, (N >> 1) - hcol, o);
        } else {
#pragma unroll
            for (int t = 0; t < 2; t++) store((int64_t)places[m] * N + col0 + 64 * t, N - (col0 + 64 * t), v[t]);
        }
    }
}

template <typename T, int BITS, int FP4, int HOLD>
__global__ void __launch_bounds__((kThreads * most_groups(HOLD)), (HOLD == rows::kTerms ? 3 : 4)) qmg_kernel(const ProductArgs a) {
    extern __shared__ __attribute__((aligned(16))) unsigned char lds[];
    const int lane = threadIdx.x & 63;
    const int N = (int)a.n;
    const int tiles = (N + kRows - 1) / kRows, experts = (int)a.experts;
    const int run = (experts + 63) >> 6, e_first = lane * run;
    auto rows_of = [&](int ei, int &begin, int &end) {
        const int rows_all = (int)a.batch;
        if (a.offsets == nullptr) {  // (one group)
            begin = 0, end = rows_all;
            return;
        }
        begin = min(max(a.offsets[ei], 0), rows_all);
        end = ei + 1 < experts ? min(max(a.offsets[ei + 1], begin), rows_all) : rows_all;
    };
    int mine = 0, kept_begin = 0, kept_end = 0;  // passes of this lane's experts; the rows of the first of them
    for (int i = 0; i < run; i++) {
        const int ei = e_first + i;
        if (ei < experts) {
            int begin, end;
            rows_of(ei, begin, end);
            if (i == 0) kept_begin = begin, kept_end = end;
            mine += (end - begin + kPassRows - 1) / kPassRows;
        }
    }
    int upto = mine;  // inclusive prefix over the lanes
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const int v = __shfl_up(upto, o);
        if (lane >= o) upto += v;
    }
    const int passes = __builtin_amdgcn_readfirstlane(__shfl(upto, 63));
    const int items = tiles * passes, per = (items + 7) >> 3;
    const int slot = (int)(blockIdx.x >> 3), item = (int)(blockIdx.x & 7) * per + slot;
    if (slot >= per || item >= items) return;  // the whole block: no barrier has been reached
    const int n0 = (item % tiles) * kRows, target = item / tiles;
    const int owner = __builtin_ctzll(__ballot(upto > target));
    int found_e = 0, found_begin = 0, found_end = 0;
    if (lane == owner) {
        int before = upto - mine;
        bool found = false;
        for (int i = 0; i < run && !found; i++) {
            const int ei = e_first + i;
            if (ei >= experts) break;
            int begin = kept_begin, end = kept_end;
            if (i > 0) rows_of(ei, begin, end);
            const int count = (end - begin + kPassRows - 1) / kPassRows;
            if (target < before + count) {
                found = true;
                found_e = ei, found_begin = begin + (target - before) * kPassRows;
                found_end = found_begin + kPassRows < end ? found_begin + kPassRows : end;
            }
            before += count;
        }
    }
    const int e = __builtin_amdgcn_readfirstlane(__shfl(found_e, owner));
    const int row_begin = __builtin_amdgcn_readfirstlane(__shfl(found_begin, owner));
    const int row_end = __builtin_amdgcn_readfirstlane(__shfl(found_end, owner));
    const int rows = row_end - row_begin;
    if (rows <= 0) return;  // the whole block: no barrier has been reached
    if (rows <= 16) run_pass<T, BITS, FP4, HOLD, 1>(a, lds, e, row_begin, rows, n0);
    else if (rows <= 32) run_pass<T, BITS, FP4, HOLD, 2>(a, lds, e, row_begin, rows, n0);
    else if (rows <= 48) run_pass<T, BITS, FP4, HOLD, 3>(a, lds, e, row_begin, rows, n0);
    else run_pass<T, BITS, FP4, HOLD, 4>(a, lds, e, row_begin, rows, n0);
}

// Affine weights that the kernels taking these products otherwise, the vector kernels, hold in float32: few pairs of a caller who ordered
// them only for speed, and off whole steps of 64 (windows of 128 of odd widths) any.  (The other kernels of several rows of one product
// round them once, and so do the sorted pairs of other callers, in two thirds of the time: 63 pairs of 4 experts of W[2880,2880], 4 bits,
// 41 us in terms, 24 rounded; of W[14336,4096], 79 and 49.)
inline bool weights_in_terms(const ProductArgs &a) { return (a.float32_weights && a.batch < 64) || a.k % (a.bits % 2 != 0 ? 128 : 64) != 0; }

// Groups of a block, by the blocks there are of one projection's `columns`: few blocks leave compute units idle and the others with a
// wavefront a SIMD (32 experts, 12 rows each, us with 1 / 2 / 4 groups: w[768,2432], 192 blocks, 8 bits 28.3 / 22.5 / 21.0, MXFP4 17.0 / 14.0 /
// 14.0; w[1536,2432], 384 blocks, MXFP4 20.8 / 20.6 / 26.4; w[2432,768], 608 blocks, 13.2 / 16.2 / 22.2).  A pair of gate and up projections
// has the groups of either, so that its sums are theirs: a pair that is not in runs of 64 rows (of an odd number of halves of 128) and
// its projections have one.  So have row-exact pairs.
inline int group_count(const ProductArgs &a, int64_t passes, int most) {
    const int64_t columns = a.glu != 0 ? a.n / 2 : a.n, blocks = columns / kRows * passes, windows = (a.k + rows::kWin - 1) / rows::kWin;
    if (a.one_group && a.k_splits > 0) return a.k_splits < most ? a.k_splits : most;
    if (a.row_exact || columns % kRows != 0) return 1;
    if (most >= 4 && windows >= 12 && blocks * 8 <= 3 * (int64_t)compute_units()) return 4;
    return windows >= 4 && blocks * 4 <= 3 * (int64_t)compute_units() ? 2 : 1;
}

template <typename T, int BITS, int FP4, int HOLD>
int32_t run_kernel(const ProductArgs &a, hipStream_t s) {
    constexpr int lds = rows::Body<T, BITS, FP4, HOLD, 4, 2, stages(4, BITS, HOLD)>::kLdsBytes;
    static_assert(lds <= 40960 && lds >= rows::Body<T, BITS, FP4, HOLD, 2, 2, stages(2, BITS, HOLD)>::kLdsBytes, "four groups a compute unit");
    static std::atomic<bool> configured{false};
    auto kernel = qmg_kernel<T, BITS, FP4, HOLD>;
    if (!configured.load()) {
        NVQ_HIP_TRY(hipFuncSetAttribute(reinterpret_cast<const void *>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, most_groups(HOLD) * lds));
        configured.store(true);
    }
    // every expert with rows adds at most one partial pass: blocks for that many items, the rest leave at once
    const int64_t met = a.experts < a.batch ? a.experts : a.batch, whole = a.batch / kPassRows;
    const int64_t items = (a.n + kRows - 1) / kRows * (whole + met);
    const int groups = group_count(a, met > whole ? met : whole, most_groups(HOLD));
    const dim3 grid((unsigned)((items + 7) / 8 * 8));
    hipLaunchKernelGGL(kernel, grid, dim3(kThreads * groups), lds * groups, s, a);
    NVQ_LAUNCH_CHECK("qmg");
    return NVQ_OK;
}

template <typename T, int BITS, int FP4>
int32_t run(const ProductArgs &a, hipStream_t s) {
    if constexpr (FP4 == rows::kAffine) {
        if (a.exact_weights) return run_kernel<T, BITS, FP4, rows::kCpu>(a, s);
        if (weights_in_terms(a)) return run_kernel<T, BITS, FP4, rows::kTerms>(a, s);
    }
    return run_kernel<T, BITS, FP4, rows::kRounded>(a, s);
}

template <int BITS, int FP4>
int32_t run_dtype(const ProductArgs &a, hipStream_t s) {
    return a.dtype == NVQ_BF16 ? run<bf16_t, BITS, FP4>(a, s) : run<f16_t, BITS, FP4>(a, s);
}

}  // namespace qmg
}  // namespace nvq
