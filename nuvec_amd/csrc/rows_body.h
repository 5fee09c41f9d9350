// The inner loop of products of a few dozen rows: a group of four wavefronts multiplies up to 16 MT rows of x with 16 NT weight rows a
// wavefront over a range of K, in windows of 128 values.  Any width of affine codes and the block formats, bfloat16 and float16, K in
// whole blocks of 32.
//
// Codes go from memory straight into the operand layout of v_mfma_f32_16x16x32: lane (row l = lane % 16, quarter q = lane / 16) loads the
// BITS dwords of its quarter of a window, several windows ahead, and K's order inside a window is permuted to suit (instruction j of a
// window takes values 8 j .. 8 j + 7 of every quarter).  x goes straight from memory into a ring of LDS stages, without a register, which
// the group shares; one barrier a window.  Scales and biases come 16 bytes a row at a time
// (8 or 16 groups) into a table of the wavefront's own in LDS.  The weights are the instruction's first operand, so that a lane's four
// sums are four consecutive weight rows of one row of x.
//
// The loads into LDS are written in assembly, unseen by the compiler's count of the loads under way; the waits at a window's start
// count the loads that are younger than the stage they wait for, and what the compiler adds for the codes only waits longer.
#pragma once

#include "qmf_kernel.h"
#include "qmv_common.h"

namespace nvq {
namespace rows {

using qmf::kAffine;
using qmf::kMxfp4;
using qmf::kMxfp8;
using qmf::kNvfp4;
using qmf::static_for;
typedef qmf::u32x4_t Piece;                                    // 16 bytes
typedef qmf::u32x2_t u32x2_a4_t __attribute__((aligned(4)));  // 8 bytes in memory at any dword

constexpr int kWaves = 4;        // of a group
constexpr int kTile = 16;        // rows of x, weight rows of a matrix instruction
constexpr int kWin = 128;        // values of K
constexpr int kXRow = 2 * kWin;  // bytes of a row of x
constexpr int kTableRow = 32;    // bytes of a weight row's part of the scales in LDS

// 16 bytes a lane from global memory straight into LDS at `lds_base` + 16 lane, unseen by the compiler's count of loads under way.
__device__ __forceinline__ void dma(const void *p, uint32_t lds_base) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off" : : "s"(lds_base), "v"(p) : "memory", "m0");
}
static __device__ const uint4 zeros = {0, 0, 0, 0};  // what x holds past the end of K

template <int BITS>
__device__ __forceinline__ void load_codes(const unsigned char *p, uint32_t (&d)[BITS]) {
    if constexpr (BITS >= 4) {
        const Piece v = *reinterpret_cast<const qmf::u32x4_a4_t *>(p);
        d[0] = v.x, d[1] = v.y, d[2] = v.z, d[3] = v.w;
    }
    if constexpr (BITS == 8) {
        const Piece v = *reinterpret_cast<const qmf::u32x4_a4_t *>(p + 16);
        d[4] = v.x, d[5] = v.y, d[6] = v.z, d[7] = v.w;
    }
    if constexpr (BITS % 4 >= 2) {
        const qmf::u32x2_t v = *reinterpret_cast<const u32x2_a4_t *>(p + BITS / 4 * 16);
        d[BITS / 4 * 4] = v.x, d[BITS / 4 * 4 + 1] = v.y;
    }
    if constexpr (BITS % 2 == 1) d[BITS - 1] = *reinterpret_cast<const uint32_t *>(p + 4 * (BITS - 1));
}

// Affine weights in float32 as terms of the element type.  With scale and bias in that type, v = code * scale + bias is a whole
// multiple of the lower one's last place, and with L bits of significand (8, 11) and their exponents close enough two terms hold it: the
// rest after one lies within 2^(E(v) - L), and its multiples fit L bits where E(v) - min(E(scale), E(bias)) <= L + 1.  float16 holds no
// multiple finer than 2^-24, so that any |v| below a half is two terms too.  Codes of `quantize` keep that by far (the bias is the
// end of the range farther from zero): two matrix instructions.  Where some lane's 32 weights do not, a third instruction brings what is
// left of v's 24 bits.  (There the range of the first term is the finite one, so that a large or infinite v is the second's; nothing is
// left then.)
template <typename T, int BITS>
__device__ __forceinline__ bool two_terms_hold(float s, float b) {
    constexpr bool bf16 = Elem<T>::code == NVQ_BF16;
    auto exponent = [](float v) { return max((int)(f2u(v) >> 23 & 255u), 1); };
    const float top = fmaxf(fabsf(b), fabsf(__builtin_fmaf((float)((1 << BITS) - 1), s, b)));
    const int high = exponent(top), low = min(s != 0.0f ? exponent(s) : 255, b != 0.0f ? exponent(b) : 255);
    if constexpr (bf16) return high - low <= 9 && top <= 3.38953139e38f;
    else return top <= 65504.0f && (high - low <= 12 || high <= 125);
}

// Piece KK of a lane's 32 affine codes as two terms; CLAMPED: of any weights, not only those that two terms hold.
template <typename T, int BITS, int KK, bool CLAMPED>
__device__ __forceinline__ void expand_terms(const uint32_t (&dw)[BITS], float s, float b, uint4 &hi, uint4 &lo) {
    constexpr float most = Elem<T>::code == NVQ_BF16 ? 3.38953139e38f : 65504.0f;
    uint32_t h[4], l[4];
    static_for<4>([&](auto i_tag) {
        constexpr int i = decltype(i_tag)::value, J = 8 * KK + 2 * i;
        const float v0 = __builtin_fmaf(qmf::code_to_float<BITS, J>(dw), s, b), v1 = __builtin_fmaf(qmf::code_to_float<BITS, J + 1>(dw), s, b);
        if constexpr (CLAMPED) h[i] = qmf::Ops<T>::pack(__builtin_amdgcn_fmed3f(v0, -most, most), __builtin_amdgcn_fmed3f(v1, -most, most));
        else h[i] = qmf::Ops<T>::pack(v0, v1);
        l[i] = qmf::Ops<T>::pack(v0 - qmf::half_lo<T>(h[i]), v1 - qmf::half_hi<T>(h[i]));
    });
    hi = make_uint4(h[0], h[1], h[2], h[3]), lo = make_uint4(l[0], l[1], l[2], l[3]);
}

// What two finite terms leave of them, exactly.
template <typename T, int BITS, int KK>
__device__ __forceinline__ uint4 left_over(const uint32_t (&dw)[BITS], float s, float b, uint4 hi, uint4 lo) {
    const uint32_t h[4] = {hi.x, hi.y, hi.z, hi.w}, l[4] = {lo.x, lo.y, lo.z, lo.w};
    uint32_t t[4];
    static_for<4>([&](auto i_tag) {
        constexpr int i = decltype(i_tag)::value, J = 8 * KK + 2 * i;
        const float v0 = __builtin_fmaf(qmf::code_to_float<BITS, J>(dw), s, b), v1 = __builtin_fmaf(qmf::code_to_float<BITS, J + 1>(dw), s, b);
        const float r0 = v0 - qmf::half_lo<T>(h[i]) - qmf::half_lo<T>(l[i]), r1 = v1 - qmf::half_hi<T>(h[i]) - qmf::half_hi<T>(l[i]);
        t[i] = qmf::Ops<T>::pack(fabsf(r0) < INFINITY ? r0 : 0.0f, fabsf(r1) < INFINITY ? r1 : 0.0f);
    });
    return make_uint4(t[0], t[1], t[2], t[3]);
}

// Weights in terms give no sum of their own to an x that is infinite or no number: it meets every term, and zero times it, or the
// difference of two infinities, is no number where the weight's product is infinite.  Of a wavefront that holds a sum that is not finite all
// such are formed anew from float32 weights and x, values k0 .. k1 - 1 of K; the finite ones stay.  (Without such a sum a look at the
// accumulators is all this costs.)
template <typename T, int BITS, int MT, int NT, class XRow, class WeightRow>
__device__ __forceinline__ void sum_plainly(const ProductArgs &a, int e, int k0, int k1, XRow xrow, WeightRow weight_row, floatx4_t (&acc)[MT][NT]) {
    bool finite = true;
#pragma unroll
    for (int m = 0; m < MT; m++)
#pragma unroll
        for (int t = 0; t < NT; t++)
#pragma unroll
            for (int i = 0; i < 4; i++) finite = finite && fabsf(acc[m][t][i]) < INFINITY;
    if (__all(finite)) return;
    const int lane = threadIdx.x & 63, l = lane & 15, q = lane >> 4, gshift = a.group == 32 ? 5 : a.group == 64 ? 6 : 7;
    const int64_t K = a.k;
    floatx4_t again[MT][NT];
#pragma unroll
    for (int m = 0; m < MT; m++)
#pragma unroll
        for (int t = 0; t < NT; t++) again[m][t] = floatx4_t{0.0f, 0.0f, 0.0f, 0.0f};
    for (int from = k0; from < k1; from += 16) {  // (whole blocks of 32)
        const int k = from + 4 * q;
        float xv[MT][4], wv[NT][4];
#pragma unroll
        for (int m = 0; m < MT; m++) {
            const T *row = (const T *)a.x + xrow(kTile * m + l) * K;
#pragma unroll
            for (int j = 0; j < 4; j++) xv[m][j] = Elem<T>::load(row, k + j);
        }
#pragma unroll
        for (int t = 0; t < NT; t++) {
            const int64_t row = (int64_t)e * a.n + weight_row(t, l), g = row * (K >> gshift) + (k >> gshift);
            const uint32_t *word = (const uint32_t *)a.w + row * (K / 32 * BITS) + (int64_t)k * BITS / 32;
            const int bit = k % 32 * BITS % 32;
            uint64_t codes = word[0];
            if (bit + 4 * BITS > 32) codes |= (uint64_t)word[1] << 32;  // (a row ends with a dword)
            const float s = Elem<T>::load((const T *)a.scales, g), b = Elem<T>::load((const T *)a.biases, g);
#pragma unroll
            for (int j = 0; j < 4; j++) wv[t][j] = __builtin_fmaf((float)((uint32_t)(codes >> (bit + BITS * j)) & ((1u << BITS) - 1u)), s, b);
        }
#pragma unroll
        for (int j = 0; j < 4; j++)
#pragma unroll
            for (int m = 0; m < MT; m++)
#pragma unroll
                for (int t = 0; t < NT; t++) again[m][t] = __builtin_amdgcn_mfma_f32_16x16x4f32(wv[t][j], xv[m][j], again[m][t], 0, 0, 0);
    }
#pragma unroll
    for (int m = 0; m < MT; m++)
#pragma unroll
        for (int t = 0; t < NT; t++)
#pragma unroll
            for (int i = 0; i < 4; i++) acc[m][t][i] = fabsf(acc[m][t][i]) < INFINITY ? acc[m][t][i] : again[m][t][i];
}

// How affine weights are held: rounded once to the element type, as nuvec's CPU product holds them (qmf::affine_pair), or as terms.
enum Hold { kRounded, kCpu, kTerms };

template <typename T, int BITS, int FP4, int HOLD, int MT, int NT, int STAGES>
struct Body {
    static constexpr int kAhead = BITS <= 4 && HOLD != kTerms ? 4 : 2;  // windows of codes under way
    static constexpr int kX = MT;  // loads of x of a window and wavefront, four rows each
    static constexpr int kXStage = MT * kTile * kXRow;
    static constexpr int kKinds = FP4 ? 1 : 2, kScaleBytes = FP4 ? 1 : 2, kPart = 16 / kScaleBytes;  // groups of a part of the scales
    static constexpr int kTablePieces = kKinds * NT * kTile * 2, kTableLoads = (kTablePieces + 63) / 64;
    static constexpr int kTableBytes = 16 * kTablePieces;  // of a wavefront
    static constexpr int kLdsBytes = STAGES * kXStage + kWaves * kTableBytes;
    static_assert(STAGES >= 2 && STAGES <= kAhead + 1, "the waits below count these loads");

    // `xrow(r)`: the row of x behind row r; `weight_row(t, r)`: row r of this wavefront's tile t, rows from `n0`, a row of the weight, on.  The range [k_begin, k1) begins at
    // a whole window and ends at one or at K; `turns` is the most windows of any group of the block.
    template <class XRow, class WeightRow>
    static __device__ __forceinline__ void run(const ProductArgs &a, unsigned char *lds, int wave, int e, int n0, int k_begin, int k1, int turns, XRow xrow,
                                               WeightRow weight_row, floatx4_t (&acc)[MT][NT]) {
        const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) unsigned char *)lds;
        const int lane = threadIdx.x & 63, l = lane & 15, q = lane >> 4;
        const int K = (int)a.k, N = (int)a.n;
        const int gshift = FP4 == kNvfp4 ? 4 : FP4 ? 5 : (a.group == 32 ? 5 : a.group == 64 ? 6 : 7);
        const int kgroups = K >> gshift;
        const uint32_t row_bytes = (uint32_t)(K >> 5) * (4 * BITS);
        const int windows = k1 > k_begin ? (k1 - k_begin + kWin - 1) / kWin : 0;
        const int k0 = windows > 0 ? k_begin : 0;  // (a group without a window asks for its rows' first values)
        int64_t xrows[kX];  // (asked for first: what is loaded after does not wait for them)
#pragma unroll
        for (int i = 0; i < kX; i++) xrows[i] = xrow(4 * (wave + kWaves * i) + (lane >> 4));
        __builtin_amdgcn_sched_barrier(0);
        unsigned char *table = lds + STAGES * kXStage + wave * kTableBytes;

        // Codes: lane (row l, quarter q) owns the 32 codes of its quarter of a window.
        const unsigned char *wbase = (const unsigned char *)a.w + ((int64_t)e * N + n0) * row_bytes + (int64_t)(k0 >> 5) * (4 * BITS);
        uint32_t woff[NT];
#pragma unroll
        for (int t = 0; t < NT; t++) woff[t] = (uint32_t)(weight_row(t, l) - n0) * row_bytes + 4 * BITS * q;
        uint32_t ring[kAhead][NT][BITS];
        // (every load is issued on every path, past the end for first values that are not used: the waits count them; a quarter past the
        // end of K repeats the window's first, and its scale and bias are zero)
        auto load_w = [&](int win, auto slot_tag) __attribute__((always_inline)) {
            constexpr int slot = decltype(slot_tag)::value;
            const int k = k0 + win * kWin + 32 * q;
            const uint32_t at = (uint32_t)(win * (16 * BITS)) - (k < K ? 0 : 4 * BITS * q);
#pragma unroll
            for (int t = 0; t < NT; t++) load_codes<BITS>(wbase + (win < windows ? woff[t] + at : 0), ring[slot][t]);
        };
        // Scales (and biases): 16 bytes of a row at a time, in the two aligned pieces that hold them.
        uintptr_t tsrc[kTableLoads], tlast[kTableLoads];
        Piece tl[kTableLoads];
        auto group_row = [&](int kind, int t, int r) {
            return (uintptr_t)(kind ? a.biases : a.scales) + (uintptr_t)((int64_t)e * N + weight_row(t, r)) * (uint32_t)(kgroups * kScaleBytes);
        };
        const int part0 = (k0 >> gshift) / kPart, part_windows = (kPart << gshift) / kWin;
#pragma unroll
        for (int j = 0; j < kTableLoads; j++) {
            const int piece = (64 * j + lane) % kTablePieces, kind = piece / (NT * kTile * 2), row = piece % (NT * kTile * 2) / 2;
            tlast[j] = ((uintptr_t)(kKinds == 2 && kind ? a.biases : a.scales) + (uintptr_t)(a.experts > 0 ? a.experts * N : N) * (uint32_t)(kgroups * kScaleBytes) - 1) & ~(uintptr_t)15;
            tsrc[j] = (group_row(kKinds == 2 ? kind : 0, row / kTile, row % kTile) & ~(uintptr_t)15) + 16 * (piece & 1);
        }
        auto load_table = [&](int part) __attribute__((always_inline)) {
#pragma unroll
            for (int j = 0; j < kTableLoads; j++) {
                const uintptr_t p = tsrc[j] + 16 * (uintptr_t)part;
                tl[j] = *reinterpret_cast<const Piece *>(p < tlast[j] ? p : tlast[j]);
            }
        };
        auto store_table = [&]() __attribute__((always_inline)) {
#pragma unroll
            for (int j = 0; j < kTableLoads; j++)
                if (kTablePieces % 64 == 0 || 64 * j + lane < kTablePieces) *reinterpret_cast<Piece *>(table + 1024 * j + 16 * lane) = tl[j];
        };
        int tread[NT][kKinds];
#pragma unroll
        for (int t = 0; t < NT; t++)
#pragma unroll
            for (int kind = 0; kind < kKinds; kind++) tread[t][kind] = ((kind * NT + t) * kTile + l) * kTableRow + (int)(group_row(kind, t, l) & 15);

        // x: piece c of row r holds values [8 (c ^ r), ...) of the row's window; past the end of K zeros.
        const T *xsrc[kX];
        int xkey[kX];
        auto place_x = [&]() __attribute__((always_inline)) {
#pragma unroll
            for (int i = 0; i < kX; i++) {
                xkey[i] = 8 * ((lane & 15) ^ ((4 * wave + (lane >> 4)) & 15));
                xsrc[i] = (const T *)a.x + xrows[i] * K + k0 + xkey[i];
            }
        };
        auto issue_x = [&](int win, int stage) __attribute__((always_inline)) {
            const bool tail = k0 + (win + 1) * kWin > K;
#pragma unroll
            for (int i = 0; i < kX; i++) {
                const void *p = xsrc[i] + win * kWin;
                if (tail) p = k0 + win * kWin + xkey[i] < K ? p : (const void *)&zeros;
                dma(p, lds0 + stage * kXStage + 1024 * (wave + kWaves * i));
            }
        };
        using S = std::conditional_t<FP4 != 0, uint8_t, T>;
        const float factor = FP4 == kNvfp4 && a.global_scale != nullptr ? ftz(a.global_scale[e] / (448.0f * 6.0f)) : 1.0f;

        load_table(part0);
        static_for<kAhead>([&](auto i) { load_w(decltype(i)::value, i); });
        __builtin_amdgcn_sched_barrier(0);
        place_x();
        static_for<STAGES - 1>([&](auto i) {
            if (decltype(i)::value < windows) issue_x(decltype(i)::value, decltype(i)::value);
        });
        constexpr int kCodeLoads = NT;  // of a window, at least
        constexpr int kYounger = (STAGES - 2) * (kX + kCodeLoads) + kCodeLoads;
        int until_part = part_windows - (k0 / kWin) % part_windows, part = part0;
        store_table();
        load_table(part + 1);
        int stage = 0;
        for (int w0 = 0; w0 < turns; w0 += kAhead) {
            static_for<kAhead>([&](auto d_tag) __attribute__((always_inline)) {
                constexpr int d = decltype(d_tag)::value;
                const int win = w0 + d;
                if (win >= turns) return;
                if (win >= STAGES && win + STAGES - 1 < windows) asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" : : "n"(kYounger) : "memory");
                else asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
                asm volatile("s_barrier" ::: "memory");
                if (win < windows) {
                    if (until_part == 0) {
                        until_part = part_windows;
                        store_table();
                        load_table(++part + 1);
                    }
                    until_part--;
                    if (win + STAGES - 1 < windows) issue_x(win + STAGES - 1, stage == 0 ? STAGES - 1 : stage - 1);
                    const unsigned char *xs = lds + stage * kXStage;
                    float scale[NT][2], bias[NT];
                    const int k = k0 + win * kWin + 32 * q;
                    const int gi = ((k >> gshift) & (kPart - 1)) * kScaleBytes;
                    const bool inside = k < K;
#pragma unroll
                    for (int t = 0; t < NT; t++) {
                        const unsigned char *ts = table + tread[t][0] + gi;
                        if constexpr (FP4 == kNvfp4) {
                            scale[t][0] = qmf::nvfp4_scale(ts[0], factor);
                            scale[t][1] = qmf::nvfp4_scale(ts[1], factor);
                            bias[t] = 0.0f;
                        } else if constexpr (FP4) {
                            scale[t][0] = scale[t][1] = ftz(e8m0_to_f32(ts[0]));
                            bias[t] = 0.0f;
                        } else {
                            scale[t][0] = scale[t][1] = Elem<T>::load(reinterpret_cast<const S *>(ts), 0);
                            bias[t] = Elem<T>::load(reinterpret_cast<const S *>(table + tread[t][kKinds - 1] + gi), 0);
                        }
                        if (!inside) scale[t][0] = scale[t][1] = bias[t] = 0.0f;
                    }
                    bool held = true;
                    if constexpr (HOLD == kTerms) {
#pragma unroll
                        for (int t = 0; t < NT; t++) held = held && two_terms_hold<T, BITS>(scale[t][0], bias[t]);
                        held = __all(held);
                    }
                    static_for<4>([&](auto j_tag) __attribute__((always_inline)) {
                        constexpr int j = decltype(j_tag)::value;
                        uint4 xf[MT], w[NT];
#pragma unroll
                        for (int m = 0; m < MT; m++) xf[m] = *reinterpret_cast<const uint4 *>(xs + (kTile * m + l) * kXRow + 16 * ((4 * q + j) ^ l));
#pragma unroll
                        for (int t = 0; t < NT; t++) {
                            if constexpr (HOLD == kTerms) {
                                uint4 lo;
                                if (held) {
                                    expand_terms<T, BITS, j, false>(ring[d][t], scale[t][0], bias[t], w[t], lo);
                                } else {
                                    expand_terms<T, BITS, j, true>(ring[d][t], scale[t][0], bias[t], w[t], lo);
                                    const uint4 rest = left_over<T, BITS, j>(ring[d][t], scale[t][0], bias[t], w[t], lo);
#pragma unroll
                                    for (int m = 0; m < MT; m++) acc[m][t] = Mfma16<T>::run(rest, xf[m], acc[m][t]);
                                }
#pragma unroll
                                for (int m = 0; m < MT; m++) acc[m][t] = Mfma16<T>::run(lo, xf[m], acc[m][t]);
                            } else {
                                w[t] = qmf::expand_piece<T, BITS, FP4, j, HOLD == kCpu>(ring[d][t], scale[t][j >> 1], bias[t]);
                            }
                        }
#pragma unroll
                        for (int m = 0; m < MT; m++)
#pragma unroll
                            for (int t = 0; t < NT; t++) acc[m][t] = Mfma16<T>::run(w[t], xf[m], acc[m][t]);
                    });
                    stage = stage == STAGES - 1 ? 0 : stage + 1;
                }
                load_w(win + kAhead, d_tag);
            });
        }
    }
};

}  // namespace rows
}  // namespace nvq
