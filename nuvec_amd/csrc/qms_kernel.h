// Products of a few dozen rows with K split over wavefronts and blocks: y[M,N] = x[M,K] . dequantize(w[N,K])^T in bfloat16 and
// float16, affine codes of 2 to 8 bits, MXFP4, MXFP8 and NVFP4, K in whole blocks of 32 (reference: crates/nuvec-core/src/kernels.rs:
// 1091-1142).  Weights are those of qmf_kernel.h: rounded once to the element type, or the CPU's (EXACT).
//
// A group of QW wavefronts (four, or one) shares the rows of x, up to 64, each wavefront 16 NT weight rows of its own, and takes K by
// turns of 256 values with the other groups of the block; K is split over the grid too where the blocks are few.  The sums of the groups
// meet in LDS, those of the splits in a second kernel.  A wavefront brings the codes of a turn in chunks of 16 bytes, consecutive
// lanes consecutive chunks, a whole turn ahead in registers, and passes them through a piece of LDS of its own into the operand
// layout of v_mfma_f32_16x16x32; scales and biases come per lane, a turn ahead, and reach the step that needs them by a lane
// exchange.  x goes through two LDS stages of 64 values a group; one barrier a step, and none where a group is one wavefront.
//
// What bounds it: a wavefront's own chain, 0.28 us a step alone on its SIMD of which the exchange, the expansion of the codes, x,
// codes and scales take a tenth to a fifth each, and beyond four wavefronts a SIMD the codes' way from memory (3.5 TB/s).  Of
// 1078 products of 3 to 400 rows that qmf_kernel or qmm_kernel took it takes 0.75 of the time, us before -> after: 17
// rows, W[2112,13568] of MXFP4 20.6 -> 12.3; 31 rows, W[404,13792] of NVFP4 30 -> 11; 62 rows, W[2560,11072] of 3 bits 35 -> 21; 16 rows,
// W[4096,11008] of 8 bits in groups of 32 26 -> 18.6; 9 rows, W[18734,1600] of 8 bits 18.6 -> 13.1.  Four steps of x ahead instead of two
// changed nothing.
#pragma once

#include "qmf_kernel.h"
#include "qmv_common.h"

namespace nvq {
namespace qms {

using qmf::static_for;

constexpr int kTile = 16;   // rows of x, weight rows of a matrix instruction
constexpr int kStep = 64;   // values of K between two barriers
constexpr int kSpan = 256;  // values of K that a group of four wavefronts takes at a time

// The shapes there are, and the most groups of one: what registers (128 of them for sixteen wavefronts) leave room for.
constexpr bool has_shape(int mt, int nt, int qw) { return qw == 4 ? nt == 1 || mt > 1 : mt * nt <= 2; }
constexpr int most_groups(int mt, int nt, int qw) { return (mt * nt <= 2 ? 16 : 8) / qw; }
constexpr int lds_bytes(int bits, int mt, int nt, int qw, int groups) {
    const int stage = kTile * mt * kStep * 2, codes = kTile * nt * (kSpan * bits / 8 + 16), part = mt * nt * 4 * 64 * qw * 4;
    const int run = groups * (2 * stage + qw * codes), end = (groups - 1) * part;
    return run > end ? run : end;
}

// QW wavefronts of a group share x, each with its own weight rows.
template <int BITS, int MT, int NT, int QW>
struct Shape {
    static constexpr int kThreads = 64 * QW, kRows = kTile * MT;
    static constexpr int kChunks = kSpan * BITS / 128;               // of 16 bytes, of a weight row in a span
    static constexpr int kAll = kTile * NT * kChunks, kLoads = (kAll + 63) / 64;
    static constexpr int kCodeRow = kSpan * BITS / 8 + 16;           // bytes between two weight rows of a span in LDS
    static constexpr int kCodeBytes = kTile * NT * kCodeRow;         // of a wavefront
    static constexpr int kStageBytes = kRows * kStep * 2;
    static constexpr int kGroupBytes = 2 * kStageBytes + QW * kCodeBytes;
    static constexpr int kPieces = (kRows * 8 + kThreads - 1) / kThreads;  // of eight values of x, a thread and step
};

template <typename T> __device__ __forceinline__ float activated(int glu_kind, float g, float up, float alpha, float limit) {
    return glu_kind == 1 + NVQ_GLU_SWIGLU       ? glu<T, NVQ_GLU_SWIGLU>(g, up, alpha, limit)
           : glu_kind == 1 + NVQ_GLU_SWIGLU_OAI ? glu<T, NVQ_GLU_SWIGLU_OAI>(g, up, alpha, limit)
                                                : glu<T, NVQ_GLU_GEGLU>(g, up, alpha, limit);
}

template <typename T, int BITS, int FP4, bool EXACT, int MT, int NT, int QW>
__global__ void __launch_bounds__((64 * QW * most_groups(MT, NT, QW))) qms_kernel(const ProductArgs a) {
    using S = Shape<BITS, MT, NT, QW>;
    using Scale = std::conditional_t<FP4 != 0, uint8_t, T>;
    constexpr bool kAffine = FP4 == qmf::kAffine, kNv = FP4 == qmf::kNvfp4;
    constexpr int kScales = kNv ? 4 : 2;  // of 64 values
    extern __shared__ __attribute__((aligned(16))) unsigned char lds_all[];
    const int groups = __builtin_amdgcn_readfirstlane(blockDim.x / S::kThreads);
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), group = wave / QW;
    const int tid = threadIdx.x & (S::kThreads - 1), lane = tid & 63, quarter = wave & (QW - 1);
    const int l = lane & 15, q = lane >> 4;
    const int M = (int)a.m, N = (int)a.n, K = (int)a.k;
    const int gshift = kNv ? 4 : FP4 ? 5 : (a.group == 32 ? 5 : a.group == 64 ? 6 : 7);
    const int kgroups = K >> gshift, kwords = K / 32 * BITS;
    const int m0 = blockIdx.y * S::kRows, n0 = blockIdx.x / (4 / QW) * (64 * NT) + blockIdx.x % (4 / QW) * (kTile * QW);
    const int k0 = blockIdx.z * a.k_split_steps * kSpan;
    const int k1 = a.k_splits > 1 && K - k0 > a.k_split_steps * kSpan ? k0 + a.k_split_steps * kSpan : K;
    unsigned char *lds = lds_all + group * S::kGroupBytes, *code_lds = lds + 2 * S::kStageBytes + quarter * S::kCodeBytes;
    // weight row `r` of tile t of this wavefront: a gate row and its up row, 64 apart, are two tiles of one lane
    auto weight_row = [&](int t, int r) { const int n = n0 + 64 * t + kTile * quarter + r; return n < N ? n : N - 1; };

    // x (rows past the end repeat the last one and are not stored; values past the end of K are zero)
    typedef qmf::u32x4_t Piece;
    Piece xs[2][S::kPieces];
    const int xr = tid >> 3, xc = tid & 7;
    const T *xrow[S::kPieces];
#pragma unroll
    for (int u = 0; u < S::kPieces; u++) {
        const int row = m0 + xr + 8 * QW * u;
        xrow[u] = (const T *)a.x + (int64_t)(row < M ? row : M - 1) * K;
    }
    // step `i` of the group's turn at k and, from 4 on, of the following ones
    auto step_at = [&](int k, int i) { return k + kSpan * groups * (i >> 2) + kStep * (i & 3); };
    auto load_x = [&](int k, auto set_tag) __attribute__((always_inline)) {
        constexpr int set = decltype(set_tag)::value;
        k += 8 * xc;
        k = k < k1 ? k : 0;
#pragma unroll
        for (int u = 0; u < S::kPieces; u++) xs[set][u] = *reinterpret_cast<const Piece *>(xrow[u] + k);
    };
    auto store_x = [&](int k, int stage, auto set_tag) __attribute__((always_inline)) {
        constexpr int set = decltype(set_tag)::value;
        const bool inside = k + 8 * xc < k1;
#pragma unroll
        for (int u = 0; u < S::kPieces; u++) {
            const int row = xr + 8 * QW * u;
            const Piece v = inside ? xs[set][u] : Piece{0, 0, 0, 0};
            if (S::kRows >= 8 * QW || row < S::kRows)
                *reinterpret_cast<Piece *>(lds + stage * S::kStageBytes + row * (kStep * 2) + ((xc ^ ((row >> 1) & 7)) * 16)) = v;
        }
    };
    // Codes.  Where K ends inside a chunk the 16 bytes up to its end are brought and moved into place; past it come a row's first bytes,
    // and zeros are stored.
    qmf::u32x4_t cw[S::kLoads];
    auto chunk_of = [&](int i) { const int c = i * 64 + lane; return (i + 1) * 64 <= S::kAll || c < S::kAll ? c : 0; };
    auto load_codes = [&](int k) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < S::kLoads; i++) {
            const int c = chunk_of(i), row = c / S::kChunks;
            int at = k / 32 * BITS + 4 * (c % S::kChunks);
            at = at >= kwords ? 0 : at + 4 > kwords ? kwords - 4 : at;
            cw[i] = *reinterpret_cast<const qmf::u32x4_a4_t *>((const uint32_t *)a.w + (int64_t)weight_row(row / kTile, row % kTile) * kwords + at);
        }
    };
    auto store_codes = [&](int k) __attribute__((always_inline)) {
        if (k + kSpan > K) {
#pragma unroll
            for (int i = 0; i < S::kLoads; i++) {
                const int missing = k / 32 * BITS + 4 * (chunk_of(i) % S::kChunks) + 4 - kwords;  // dwords past the end
                qmf::u32x4_t &v = cw[i];
                v = missing >= 4   ? qmf::u32x4_t{0, 0, 0, 0}
                    : missing == 3 ? qmf::u32x4_t{v.w, 0, 0, 0}
                    : missing == 2 ? qmf::u32x4_t{v.z, v.w, 0, 0}
                    : missing == 1 ? qmf::u32x4_t{v.y, v.z, v.w, 0}
                                   : v;
            }
        }
#pragma unroll
        for (int i = 0; i < S::kLoads; i++) {
            const int c = i * 64 + lane;
            if ((i + 1) * 64 <= S::kAll || c < S::kAll)
                *reinterpret_cast<qmf::u32x4_t *>(code_lds + (c / S::kChunks) * S::kCodeRow + (c % S::kChunks) * 16) = cw[i];
        }
        __builtin_amdgcn_wave_barrier();  // (the wavefront's LDS accesses execute in order)
    };
    // The eight codes of this lane for block b (of 32) of step j.
    auto codes_of = [&](int t, int j, int b) __attribute__((always_inline)) {
        const uint32_t *row = reinterpret_cast<const uint32_t *>(code_lds + (t * kTile + l) * S::kCodeRow) + (2 * j + b) * BITS;
        if constexpr (BITS == 4) return (uint64_t)row[q];
        else if constexpr (BITS == 8) return *reinterpret_cast<const uint64_t *>(row + 2 * q);
        else {
            const int first = q * BITS / 4, bit = 8 * (q * BITS % 4);
            uint64_t v = row[first];
            if constexpr (BITS > 2) v |= (uint64_t)row[first + 1 < BITS ? first + 1 : BITS - 1] << 32;
            return v >> bit;
        }
    };
    // Scales and biases of a turn: lane (q, l) brings those of step q for weight row l of each tile.
    Scale sn[NT][kScales], bn[NT][kAffine ? 2 : 1];
    uint32_t sw[NT], bw[NT];
    auto load_scales = [&](int k) __attribute__((always_inline)) {
#pragma unroll
        for (int t = 0; t < NT; t++)
#pragma unroll
            for (int b = 0; b < kScales; b++) {
                const int at = k + kStep * q + b * (kNv ? 16 : 32);
                const int64_t g = (int64_t)weight_row(t, l) * kgroups + (at < k1 ? at >> gshift : 0);
                sn[t][b] = ((const Scale *)a.scales)[g];
                if constexpr (kAffine) bn[t][b] = ((const Scale *)a.biases)[g];
            }
    };
    // (past the end of K: zero)
    auto take_scales = [&](int k) __attribute__((always_inline)) {
        const uint32_t keep = (k + kStep * q < k1 ? (kNv ? 0xFFFFu : kAffine ? 0xFFFFu : 0xFFu) : 0u) | (k + kStep * q + 32 < k1 ? (kNv || kAffine ? 0xFFFF0000u : 0xFF00u) : 0u);
#pragma unroll
        for (int t = 0; t < NT; t++) {
            if constexpr (kAffine) {
                sw[t] = (uint32_t)__builtin_bit_cast(uint16_t, sn[t][0]) | (uint32_t)__builtin_bit_cast(uint16_t, sn[t][1]) << 16;
                sw[t] &= keep;
                bw[t] = (uint32_t)__builtin_bit_cast(uint16_t, bn[t][0]) | (uint32_t)__builtin_bit_cast(uint16_t, bn[t][1]) << 16;
                bw[t] &= keep;
            } else {
                sw[t] = 0;
#pragma unroll
                for (int b = 0; b < kScales; b++) sw[t] |= (uint32_t)sn[t][b] << (8 * b);
                sw[t] &= keep;
            }
        }
    };
    const float factor = kNv ? qmf::nvfp4_factor(a, 0) : 1.0f;

    floatx4_t acc[MT][NT];
#pragma unroll
    for (int m = 0; m < MT; m++)
#pragma unroll
        for (int t = 0; t < NT; t++) acc[m][t] = floatx4_t{0.0f, 0.0f, 0.0f, 0.0f};

    // Every request is made on every path, past the end for first values that are not used: a wait for one load would otherwise be
    // a wait for all.  The groups walk the same number of turns.
    int k = k0 + group * kSpan;
    const int turns = (k1 - k0 + kSpan * groups - 1) / (kSpan * groups);
    load_codes(k);
    load_scales(k);
    static_for<2>([&](auto i) { load_x(step_at(k, i), i); });
    store_x(k, 0, std::integral_constant<int, 0>{});
    load_x(step_at(k, 2), std::integral_constant<int, 0>{});
    __syncthreads();
    for (int turn = 0; turn < turns; turn++, k += kSpan * groups) {
        store_codes(k);
        take_scales(k);
        load_codes(k + kSpan * groups);
        load_scales(k + kSpan * groups);
        static_for<4>([&](auto j_tag) {
            constexpr int j = decltype(j_tag)::value;
            constexpr std::integral_constant<int, (j + 1) & 1> set;
            const unsigned char *stage = lds + (j & 1) * S::kStageBytes;
            uint4 xo[2][MT];
#pragma unroll
            for (int b = 0; b < 2; b++)
#pragma unroll
                for (int m = 0; m < MT; m++) {
                    const int row = kTile * m + l;
                    xo[b][m] = *reinterpret_cast<const uint4 *>(stage + row * (kStep * 2) + (((4 * b + q) ^ ((row >> 1) & 7)) * 16));
                }
            uint64_t codes[2][NT];
            uint32_t sword[NT], bword[NT];
#pragma unroll
            for (int t = 0; t < NT; t++) {
                codes[0][t] = codes_of(t, j, 0), codes[1][t] = codes_of(t, j, 1);
                sword[t] = (uint32_t)__builtin_amdgcn_ds_bpermute(4 * (l + 16 * j), (int)sw[t]);
                bword[t] = kAffine ? (uint32_t)__builtin_amdgcn_ds_bpermute(4 * (l + 16 * j), (int)bw[t]) : 0u;
            }
            store_x(step_at(k, j + 1), (j + 1) & 1, set);
            load_x(step_at(k, j + 3), set);
            __builtin_amdgcn_sched_barrier(0);
            static_for<2>([&](auto b_tag) {
                constexpr int b = decltype(b_tag)::value;
#pragma unroll
                for (int t = 0; t < NT; t++) {
                    uint32_t dw[BITS] = {};
                    dw[0] = (uint32_t)codes[b][t], dw[1] = (uint32_t)(codes[b][t] >> 32);
                    float scale, bias = 0.0f;
                    if constexpr (kAffine) scale = b ? Pair<T>::hi(sword[t]) : Pair<T>::lo(sword[t]), bias = b ? Pair<T>::hi(bword[t]) : Pair<T>::lo(bword[t]);
                    else if constexpr (kNv) scale = qmf::nvfp4_scale((sword[t] >> (16 * b + 8 * (q >> 1))) & 255u, factor);
                    else scale = ftz(e8m0_to_f32((sword[t] >> (8 * b)) & 255u));
                    const uint4 w = qmf::expand_piece<T, BITS, FP4, 0, EXACT>(dw, scale, bias);
#pragma unroll
                    for (int m = 0; m < MT; m++) acc[m][t] = Mfma16<T>::run(xo[b][m], w, acc[m][t]);
                }
            });
            if constexpr (QW > 1) __syncthreads();
            else __builtin_amdgcn_wave_barrier();
        });
    }
    __syncthreads();

    // The groups' sums, added in order by the first group's threads.  Element i of a thread: tile m, tile t, element e.
    float *part = reinterpret_cast<float *>(lds_all);
    if (group > 0) {
#pragma unroll
        for (int m = 0; m < MT; m++)
#pragma unroll
            for (int t = 0; t < NT; t++)
#pragma unroll
                for (int e = 0; e < 4; e++) part[((group - 1) * MT * NT * 4 + (m * NT + t) * 4 + e) * S::kThreads + tid] = acc[m][t][e];
    }
    __syncthreads();
    if (group > 0) return;
    for (int g = 0; g < groups - 1; g++)
#pragma unroll
        for (int m = 0; m < MT; m++)
#pragma unroll
            for (int t = 0; t < NT; t++)
#pragma unroll
                for (int e = 0; e < 4; e++) acc[m][t][e] += part[(g * MT * NT * 4 + (m * NT + t) * 4 + e) * S::kThreads + tid];

    // Element e of lane (q, l): row 4 q + e of x, weight row l.
#pragma unroll
    for (int m = 0; m < MT; m++)
#pragma unroll
        for (int e = 0; e < 4; e++) {
            const int row = m0 + kTile * m + 4 * q + e, col = n0 + kTile * quarter + l;
            if (row >= M) continue;
            if (a.k_splits > 1) {
#pragma unroll
                for (int t = 0; t < NT; t++)
                    if (col + 64 * t < N) a.partials[((int64_t)blockIdx.z * M + row) * N + col + 64 * t] = acc[m][t][e];
            } else if (NT == 2 && a.glu != 0) {  // (N is whole blocks)
                const float g = add_row_bias<T>(a.row_bias, acc[m][0][e], col), up = add_row_bias<T>(a.row_bias, acc[m][NT - 1][e], col + 64);
                Elem<T>::store((T *)a.y, (int64_t)row * (N / 2) + blockIdx.x / (4 / QW) * 64 + blockIdx.x % (4 / QW) * (kTile * QW) + kTile * quarter + l,
                               activated<T>(a.glu, rounded<T>(g), rounded<T>(up), a.glu_alpha, a.glu_limit));
            } else {
#pragma unroll
                for (int t = 0; t < NT; t++)
                    if (col + 64 * t < N) Elem<T>::store((T *)a.y, (int64_t)row * N + col + 64 * t, add_row_bias<T>(a.row_bias, acc[m][t][e], col + 64 * t));
            }
        }
}

// The parts of a split K, eight under way at a time and added by pairs; then the bias, or both biases and the gated activation.
template <typename T>
__global__ void __launch_bounds__(256) qms_reduce_kernel(const ProductArgs a) {
    const int64_t total = a.m * a.n, outputs = a.glu != 0 ? total / 2 : total, i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= outputs) return;
    auto sum_at = [&](int64_t at) {
        float sum = 0.0f;
        for (int s = 0; s < a.k_splits; s += 8) {
            float v[8];
#pragma unroll
            for (int u = 0; u < 8; u++) v[u] = a.partials[(int64_t)(s + u < a.k_splits ? s + u : s) * total + at];
#pragma unroll
            for (int u = 0; u < 8; u++) v[u] = s + u < a.k_splits ? v[u] : 0.0f;
            sum += ((v[0] + v[1]) + (v[2] + v[3])) + ((v[4] + v[5]) + (v[6] + v[7]));
        }
        return sum;
    };
    if (a.glu != 0) {
        const int64_t half = a.n / 2, row = i / half, c = i % half, col = c / 64 * 128 + c % 64;
        const float g = add_row_bias<T>(a.row_bias, sum_at(row * a.n + col), col), up = add_row_bias<T>(a.row_bias, sum_at(row * a.n + col + 64), col + 64);
        Elem<T>::store((T *)a.y, i, activated<T>(a.glu, rounded<T>(g), rounded<T>(up), a.glu_alpha, a.glu_limit));
    } else {
        Elem<T>::store((T *)a.y, i, add_row_bias<T>(a.row_bias, sum_at(i), i % a.n));
    }
}

template <typename T, int BITS, int FP4, bool EXACT, int MT, int NT, int QW>
int32_t run_shape(const ProductArgs &a, const Plan &p, hipStream_t s) {
    using S = Shape<BITS, MT, NT, QW>;
    auto kernel = qms_kernel<T, BITS, FP4, EXACT, MT, NT, QW>;
    const int lds = lds_bytes(BITS, MT, NT, QW, p.groups);
    static std::atomic<bool> configured{false};
    if (lds > 64 * 1024 && !configured.load()) {
        NVQ_HIP_TRY(hipFuncSetAttribute(reinterpret_cast<const void *>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024));
        configured.store(true);
    }
    const dim3 grid((unsigned)((a.n + 64 * NT - 1) / (64 * NT) * (4 / QW)), (unsigned)((a.m + S::kRows - 1) / S::kRows), (unsigned)a.k_splits);
    hipLaunchKernelGGL(kernel, grid, dim3(S::kThreads * p.groups), lds, s, a);
    NVQ_LAUNCH_CHECK("qms");
    if (a.k_splits <= 1) return NVQ_OK;
    const int64_t outputs = a.glu != 0 ? a.m * a.n / 2 : a.m * a.n;
    hipLaunchKernelGGL((qms_reduce_kernel<T>), dim3((unsigned)((outputs + 255) / 256)), dim3(256), 0, s, a);
    NVQ_LAUNCH_CHECK("qms_reduce");
    return NVQ_OK;
}

template <typename T, int BITS, int FP4, bool EXACT>
int32_t run(const ProductArgs &a, const Plan &p, hipStream_t s) {
    switch (100 * p.mt + 10 * p.nt + p.qw) {
    case 111: return run_shape<T, BITS, FP4, EXACT, 1, 1, 1>(a, p, s);
    case 121: return run_shape<T, BITS, FP4, EXACT, 1, 2, 1>(a, p, s);
    case 114: return run_shape<T, BITS, FP4, EXACT, 1, 1, 4>(a, p, s);
    case 211: return run_shape<T, BITS, FP4, EXACT, 2, 1, 1>(a, p, s);
    case 214: return run_shape<T, BITS, FP4, EXACT, 2, 1, 4>(a, p, s);
    case 224: return run_shape<T, BITS, FP4, EXACT, 2, 2, 4>(a, p, s);
    case 414: return run_shape<T, BITS, FP4, EXACT, 4, 1, 4>(a, p, s);
    default: return run_shape<T, BITS, FP4, EXACT, 4, 2, 4>(a, p, s);
    }
}

template <int BITS, int FP4>
int32_t run_dtype(const ProductArgs &a, const Plan &p, hipStream_t s) {
    if constexpr (FP4 == qmf::kAffine)
        if (a.exact_weights) return a.dtype == NVQ_BF16 ? run<bf16_t, BITS, FP4, true>(a, p, s) : run<f16_t, BITS, FP4, true>(a, p, s);
    return a.dtype == NVQ_BF16 ? run<bf16_t, BITS, FP4, false>(a, p, s) : run<f16_t, BITS, FP4, false>(a, p, s);
}

}  // namespace qms

// One per code width, each in its own translation unit.
int32_t launch_qms_b2(const ProductArgs &a, const qms::Plan &p, hipStream_t s);
int32_t launch_qms_b3(const ProductArgs &a, const qms::Plan &p, hipStream_t s);
int32_t launch_qms_b4(const ProductArgs &a, const qms::Plan &p, hipStream_t s);
int32_t launch_qms_b5(const ProductArgs &a, const qms::Plan &p, hipStream_t s);
int32_t launch_qms_b6(const ProductArgs &a, const qms::Plan &p, hipStream_t s);
int32_t launch_qms_b8(const ProductArgs &a, const qms::Plan &p, hipStream_t s);
int32_t launch_qms_fp4(const ProductArgs &a, const qms::Plan &p, hipStream_t s);
int32_t launch_qms_fp8(const ProductArgs &a, const qms::Plan &p, hipStream_t s);
int32_t launch_qms_nvfp4(const ProductArgs &a, const qms::Plan &p, hipStream_t s);

}  // namespace nvq
