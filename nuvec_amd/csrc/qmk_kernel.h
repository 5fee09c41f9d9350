// Tiled quantized products y[M,N] = x[M,K] . dequantize(w[N,K])^T on the gfx950 matrix cores for products whose 256 x 256 tiles
// (qmm_kernel.h) would not fill the chip, and for those that take the CPU's weights: affine 1- to 6- and 8-bit codes and the block
// formats, bfloat16 and float16, K in whole blocks of 32.  Values follow nuvec's CPU product (reference:
// crates/nuvec-core/src/kernels.rs:1091-1142): weights as in qmf_kernel.h, sums in float32.
//
// A block of eight wavefronts, two a SIMD, owns 32 TI x 128 of y and walks K in windows of 128.  Each wavefront has all rows of the
// tile, 64 of its weight rows and one quarter of every window: no weight is expanded twice in a block and a fragment of x serves two
// matrix instructions (with 2 x 2 wavefronts of 64 x 64 over all of K, the kernel before, each weight was expanded twice and a SIMD had
// one wavefront).  The sums of the four quarters meet in LDS at the end.  x, the packed codes and the scales arrive by direct loads
// into three LDS stages, two windows ahead, one barrier a window; the pieces of a row's codes are those of qmm_kernel.h, scales and
// biases come 16 bytes a row at a time as in rows_body.h.  A quarter past the end of K is not multiplied, so that K needs no whole windows.
//
// What bounds it: the vector instructions of the expansion (512 rows, W[4096,4096] of 4 bits, the CPU's weights: 230 a window and
// wavefront, two wavefronts a SIMD, beside 16 matrix instructions that cost the issue 14 cycles each: 3080 cycles a window, of which the
// matrix cores are busy 1024), with half of the LDS cycles bank conflicts (scales lie 32 bytes a row apart, so that 32 lanes read a quarter of
// the banks, and the codes of rows r and r + 16 share theirs: SQ_LDS_BANK_CONFLICT 2.05e6 of SQ_LDS_IDX_ACTIVE 4.05e6); a block's first loads and
// the exchange of the sums, 5 us of a short K.  A substep's operands are prepared under
// the matrix instructions of the one before (5 % against a window's reads, expansion and products one after the other).
// us, before -> here: 445 rows, W[2150,1280] of 4 bits 22.6 -> 13.3; 46 rows, W[13247,6688] of NVFP4 49 -> 33; 66 rows, W[16212,4992] of 3
// bits 45 -> 36; 455 rows, W[8250,7360] of 3 bits 146 -> 93; 512 rows, W[4096,14336] of 4 bits 111 -> 86.
#pragma once

#include "qmm_kernel.h"
#include "rows_body.h"

namespace nvq {
namespace qmk {

using namespace qmf;  // element operations and code expansion
using qmm::dma;
using qmm::dma_wait;
using qmm::Pieces;

constexpr int kWin = 128, kQuarter = 32;  // values of K
constexpr int kWaves = 8, kThreads = 64 * kWaves, kStages = 3;
constexpr int kCols = 128, TJ = 2;        // weight rows of a block; tiles of 32 of them a wavefront
constexpr int kTableBytes = 16 * kThreads;  // scales and biases: two aligned pieces of 16 bytes of each row and kind

template <int BITS, int TI>
struct Shape {
    static constexpr int kRows = 32 * TI;
    static constexpr int kXBytes = kRows * kWin * 2;
    static constexpr int kPieceBytes = Pieces<BITS>::dwords == 1 ? 4 : 16;  // of LDS a slot, the codes of a weight row and quarter
    static constexpr int kRegionBytes = kThreads * kPieceBytes;
    static constexpr int kStageBytes = kXBytes + Pieces<BITS>::count * kRegionBytes;
    static constexpr int kLoads = TI + Pieces<BITS>::count;  // of a window and lane, without the table's
    static constexpr int kRun = kStages * kStageBytes + 2 * kTableBytes, kEnd = 4 * kWaves * 4096;  // LDS of the loop, of the sums
    static constexpr int kLdsBytes = kRun > kEnd ? kRun : kEnd;
};

template <typename T, int BITS, int FP4, bool EXACT, int TI>
__global__ void __launch_bounds__(kThreads, 2) qmk_kernel(const ProductArgs a) {
    using S = Shape<BITS, TI>;
    using P = Pieces<BITS>;
    using Scale = std::conditional_t<FP4 != 0, uint8_t, T>;
    constexpr int kKinds = FP4 ? 1 : 2, kScaleBytes = (int)sizeof(Scale), kPart = 16 / kScaleBytes;  // groups of a part of the table
    extern __shared__ __attribute__((aligned(16))) unsigned char lds[];
    const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) unsigned char *)lds;
    const int tid = threadIdx.x, lane = tid & 63, l32 = lane & 31, h = lane >> 5;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), wn = wave & 1, quarter = wave >> 1;
    const int K = (int)a.k, N = (int)a.n, M = (int)a.m;
    const int gshift = FP4 == kNvfp4 ? 4 : FP4 ? 5 : (a.group == 32 ? 5 : a.group == 64 ? 6 : 7);
    const int kgroups = K >> gshift;
    const uint32_t row_bytes = (uint32_t)(K >> 5) * (4 * BITS);
    const int m0 = blockIdx.y * S::kRows, n0 = blockIdx.x * kCols;
    int first = 0, windows = (K + kWin - 1) / kWin;
    int64_t bx = 0, bw = 0, bs = 0, by = 0;
    if (a.k_splits > 1) {  // this block's windows of K; float32 partial sums for a second kernel
        first = blockIdx.z * a.k_split_steps;
        windows = windows - first < a.k_split_steps ? windows - first : a.k_split_steps;
        if (windows <= 0) return;  // (the host sizes the grid so that every split has a window)
    } else if (a.batch > 1) {  // a batch with one stride per operand
        bx = (int64_t)blockIdx.z * a.x_strides[0], bw = (int64_t)blockIdx.z * a.w_strides[0], bs = (int64_t)blockIdx.z * a.s_strides[0];
        by = (int64_t)blockIdx.z * M * N;
    }
    const char *xbase = reinterpret_cast<const char *>((const T *)a.x + bx + (int64_t)m0 * K);
    const char *wbase = reinterpret_cast<const char *>((const uint32_t *)a.w + bw) + (int64_t)n0 * row_bytes;

    // x: load i fills the 512 slots of 16 bytes from slot 512 i on; slot s is row s / 16 and holds its chunk s % 16 ^ row % 16 of the
    // window (a row's 256 bytes are all banks: sixteen rows read one chunk from sixteen places).  Rows past the end repeat the last one,
    // chunks past the end of K the window's first.
    const int chunk = (lane & 15) ^ (tid >> 4 & 15);
    uint32_t xoff[TI];
#pragma unroll
    for (int i = 0; i < TI; i++) {
        const int row = 32 * i + (tid >> 4);
        xoff[i] = ((uint32_t)(m0 + row < M ? row : M - 1 - m0) * (uint32_t)K + 8 * chunk) * 2;
    }
    // Codes: slot s (of this thread) is weight row s / 4, quarter s % 4 ^ row / 4 % 4 (the same, for a quarter of sixteen rows).
    const int wrow = tid >> 2, wquarter = (tid & 3) ^ (wrow >> 2 & 3);
    const uint32_t woff = (uint32_t)(n0 + wrow < N ? wrow : N - 1 - n0) * row_bytes + wquarter * (4 * BITS);
    // The table: piece p is half p % 2 of row p / 2 % 128, scales, then biases (block formats: the scales twice).
    const int tkind = kKinds == 2 ? tid >> 8 : 0, trow = tid >> 1 & 127;
    auto group_row = [&](int kind, int row) {
        const char *from = reinterpret_cast<const char *>(kKinds == 2 && kind ? a.biases : a.scales);
        return (uintptr_t)from + (uintptr_t)((bs + (int64_t)(n0 + row < N ? n0 + row : N - 1) * kgroups) * kScaleBytes);
    };
    const uintptr_t tsrc = (group_row(tkind, trow) & ~(uintptr_t)15) + 16 * (tid & 1);
    const uintptr_t tlast = (group_row(tkind, N - 1 - n0) + (uintptr_t)(kgroups * kScaleBytes) - 1) & ~(uintptr_t)15;  // the piece of the last group there is
    const int part_shift = gshift + (kScaleBytes == 1 ? 4 : 3) - 7;  // log2 of a part's windows
    const uint32_t lds_wave = lds0 + wave * 1024;
    auto issue = [&](int win, int stage) __attribute__((always_inline)) {
        const int at = first + win;
        if (win == 0 || (at & ((1 << part_shift) - 1)) == 0) {  // (a part begins: its table lands with the window)
            const uintptr_t p = tsrc + 16 * (uintptr_t)(at >> part_shift);
            rows::dma(reinterpret_cast<const void *>(p < tlast ? p : tlast), lds_wave + kStages * S::kStageBytes + (at >> part_shift & 1) * kTableBytes);
        }
        const bool tail = (at + 1) * kWin > K;
        const uint32_t xback = tail && at * kWin + 8 * chunk >= K ? 16 * chunk : 0, wback = tail && at * kWin + kQuarter * wquarter >= K ? 4 * BITS * wquarter : 0;
        const uint32_t to = lds_wave + stage * S::kStageBytes;
        const char *xwin = xbase + (int64_t)at * (kWin * 2), *wwin = wbase + (int64_t)at * (16 * BITS);
#pragma unroll
        for (int i = 0; i < TI; i++) dma<4>(xwin, xoff[i] - xback, to + i * (kThreads * 16));
#pragma unroll
        for (int piece = 0; piece < P::count; piece++)
            dma<P::dwords>(wwin + piece * (P::dwords * 4), woff - wback,
                           to + S::kXBytes + piece * S::kRegionBytes - (S::kPieceBytes == 16 ? 0 : wave * 768));
    };

    // This lane's two weight rows: their codes' slots and their scales' places in a table.
    int slot[TJ], tread[TJ][kKinds];
#pragma unroll
    for (int j = 0; j < TJ; j++) {
        const int row = 64 * wn + 32 * j + l32;
        slot[j] = 4 * row + (quarter ^ (row >> 2 & 3));
#pragma unroll
        for (int kind = 0; kind < kKinds; kind++) tread[j][kind] = (kind * 128 + row) * 32 + (int)(group_row(kind, row) & 15);
    }
    // The sixteen codes of the lane's half of its quarter, in the low dwords.
    auto read_codes = [&](const unsigned char *codes, int s, uint32_t (&dw)[BITS]) __attribute__((always_inline)) {
        if constexpr (BITS == 4) {
            const uint2 v = *reinterpret_cast<const uint2 *>(codes + s * 16 + 8 * h);
            dw[0] = v.x, dw[1] = v.y;
        } else if constexpr (BITS == 8) {
            const uint4 v = *reinterpret_cast<const uint4 *>(codes + h * S::kRegionBytes + s * 16);
            dw[0] = v.x, dw[1] = v.y, dw[2] = v.z, dw[3] = v.w;
        } else if constexpr (BITS == 6) {
            const uint32_t *v = reinterpret_cast<const uint32_t *>(codes + h * S::kRegionBytes + s * 16);
            dw[0] = v[0], dw[1] = v[1], dw[2] = v[2];
        } else if constexpr (BITS == 5) {
            const uint32_t *v = reinterpret_cast<const uint32_t *>(codes + 2 * h * S::kRegionBytes) + s;
            const uint32_t d0 = v[0], d1 = v[S::kRegionBytes / 4], d2 = v[2 * S::kRegionBytes / 4];
            dw[0] = __builtin_amdgcn_alignbit(d1, d0, 16 * h), dw[1] = __builtin_amdgcn_alignbit(d2, d1, 16 * h), dw[2] = d2 >> (16 * h);
        } else if constexpr (BITS == 3) {
            const uint32_t *v = reinterpret_cast<const uint32_t *>(codes + s * 16) + h;
            const uint32_t d0 = v[0], d1 = v[1];
            dw[0] = __builtin_amdgcn_alignbit(d1, d0, 16 * h), dw[1] = d1 >> (16 * h);
        } else if constexpr (BITS == 2) {
            dw[0] = reinterpret_cast<const uint32_t *>(codes + h * S::kRegionBytes)[s];
        } else {
            dw[0] = reinterpret_cast<const uint32_t *>(codes)[s] >> (16 * h);
        }
    };
    const float factor = FP4 == kNvfp4 ? nvfp4_factor(a, 0) : 1.0f;  // (one matrix, or a batch that shares the scale)

    floatx16_t acc[TI][TJ];
#pragma unroll
    for (int i = 0; i < TI; i++)
#pragma unroll
        for (int j = 0; j < TJ; j++)
#pragma unroll
            for (int e = 0; e < 16; e++) acc[i][j][e] = 0.0f;

    // The codes and scales of this lane's columns for window `win`, as read; converted where first used.
    uint32_t dw[TJ][BITS];
    Scale sraw[TJ], braw[TJ];
    float scale[TJ], bias[TJ];
    auto read_window = [&](int win, int stage) __attribute__((always_inline)) {
        const unsigned char *codes = lds + stage * S::kStageBytes + S::kXBytes;
        const unsigned char *table = lds + kStages * S::kStageBytes + ((first + win) >> part_shift & 1) * kTableBytes;
        const int k = (first + win) * kWin + kQuarter * quarter + (FP4 == kNvfp4 ? 16 * h : 0), group = ((k >> gshift) & (kPart - 1)) * kScaleBytes;
#pragma unroll
        for (int j = 0; j < TJ; j++) {
            read_codes(codes, slot[j], dw[j]);
            sraw[j] = *reinterpret_cast<const Scale *>(table + tread[j][0] + group);
            if constexpr (!FP4) braw[j] = *reinterpret_cast<const Scale *>(table + tread[j][kKinds - 1] + group);
        }
    };
    // What prepares substep U of a window into buffer U, in items: fragments of x are read and dwords of weights expanded by turns, for a
    // window's first substep all reads first (its codes were only just requested).
    uint4 af[2][TI], bf[2][TJ];
    constexpr int kItems = TI + 4 * TJ, kMfmas = TI * TJ;
    auto side_item = [&](int stage, auto u_tag, auto t_tag) __attribute__((always_inline)) {
        constexpr int U = decltype(u_tag)::value, t = decltype(t_tag)::value;
        constexpr bool alternate = U != 0 && t < 2 * TI, is_read = alternate ? t % 2 == 0 : U == 0 && t < TI;
        constexpr int index = alternate ? t / 2 : is_read ? t : t - TI;
        if constexpr (is_read) {
            const int row = 32 * index + l32;
            af[U][index] = *reinterpret_cast<const uint4 *>(lds + stage * S::kStageBytes + row * (kWin * 2) + (((4 * quarter + 2 * h + U) ^ (row & 15)) << 4));
        } else {
            constexpr int j = index / 4, d = index % 4;
            if constexpr (U == 0 && d == 0) {
                if constexpr (FP4 == kNvfp4) scale[j] = nvfp4_scale(sraw[j], factor);
                else if constexpr (FP4) scale[j] = ftz(e8m0_to_f32(sraw[j]));
                else scale[j] = Elem<T>::load(&sraw[j], 0);
                bias[j] = 0.0f;
                if constexpr (!FP4) bias[j] = Elem<T>::load(&braw[j], 0);
            }
            const uint32_t v = qmm::expand_dword<T, BITS, FP4, U, d, EXACT>(dw[j], scale[j], bias[j]);
            if constexpr (d == 0) bf[U][j].x = v;
            else if constexpr (d == 1) bf[U][j].y = v;
            else if constexpr (d == 2) bf[U][j].z = v;
            else bf[U][j].w = v;
        }
    };
    using First = std::integral_constant<int, 0>;
    using Second = std::integral_constant<int, 1>;
    issue(0, 0);
    if (windows > 1) issue(1, 1);
    if (windows > 1) dma_wait<S::kLoads>();
    else dma_wait<0>();
    __syncthreads();
    read_window(0, 0);
    static_for<kItems>([&](auto t) { side_item(0, First{}, t); });
    int stage = 0;
    for (int win = 0; win < windows; win++) {
        // Entering: the window is visible to everyone, this lane holds its codes, buffer 0 its first substep, and everyone is done with
        // the window before, whose stage the loads refill.
        const int stage1 = stage == kStages - 1 ? 0 : stage + 1;
        const bool live = (first + win) * kWin + kQuarter * quarter < K;  // (this wavefront's last window may lie past the end)
        if (win + 2 < windows) issue(win + 2, stage1 == kStages - 1 ? 0 : stage1 + 1);
        auto multiply = [&](auto u_tag, auto next_tag, int from) __attribute__((always_inline)) {
            constexpr int u = decltype(u_tag)::value;
            static_for<kMfmas>([&](auto q_tag) __attribute__((always_inline)) {
                constexpr int q = decltype(q_tag)::value, i = q % TI, j = q / TI;
                acc[i][j] = Ops<T>::mfma(af[u][i], bf[u][j], acc[i][j]);
                static_for<kItems>([&](auto t_tag) __attribute__((always_inline)) {
                    constexpr int t = decltype(t_tag)::value;
                    if constexpr (t >= q * kItems / kMfmas && t < (q + 1) * kItems / kMfmas) side_item(from, next_tag, t_tag);
                });
                qmm::pin();
            });
        };
        if (live) multiply(First{}, Second{}, stage);
        // the next window has landed, everyone's, and everyone has read the last of this one
        if (win + 2 < windows) dma_wait<S::kLoads>();
        else dma_wait<0>();
        __syncthreads();
        if (live) {
            read_window(win + 1, stage1);
            qmm::pin();
            multiply(Second{}, First{}, stage1);
        }
        stage = stage1;
    }

    // The quarters' sums: a round of four tiles of 32 x 32 for each half of the weight rows, every wavefront's through LDS; wavefront
    // (wn, q) adds up and stores tile q of the round.
    float *sums = reinterpret_cast<float *>(lds);
#pragma unroll
    for (int round = 0; round < TI * TJ / 4; round++) {
        __syncthreads();
#pragma unroll
        for (int t = 0; t < 4; t++) {
            const int i = TI == 4 ? t : t & 1, j = TI == 4 ? round : t >> 1;
#pragma unroll
            for (int e = 0; e < 16; e++) sums[(((wn * 4 + t) * 4 + quarter) * 16 + e) * 64 + lane] = acc[i][j][e];
        }
        __syncthreads();
        const int i = TI == 4 ? quarter : quarter & 1, j = TI == 4 ? round : quarter >> 1;
        float v[16];
#pragma unroll
        for (int e = 0; e < 16; e++) {
            const float *p = sums + ((wn * 4 + quarter) * 64 + e) * 64 + lane;
            v[e] = (p[0] + p[16 * 64]) + (p[2 * 16 * 64] + p[3 * 16 * 64]);
        }
        // Element e of a 32 x 32 tile is row 8 (e / 4) + 4 (lane / 32) + e % 4, column lane % 32.
        const int col = n0 + 64 * wn + 32 * j + l32, row0 = m0 + 32 * i + 4 * h;
        if (col < N) {
            if (a.k_splits > 1) {
                float *out = a.partials + ((int64_t)blockIdx.z * M + row0) * N + col;
#pragma unroll
                for (int e = 0; e < 16; e++) {
                    const int r = 8 * (e >> 2) + (e & 3);
                    if (row0 + r < M) out[(int64_t)r * N] = v[e];
                }
            } else {
                uint16_t *out = reinterpret_cast<uint16_t *>((T *)a.y + by) + (int64_t)row0 * N + col;
#pragma unroll
                for (int e = 0; e < 16; e += 2) {
                    const uint32_t pair = Ops<T>::pack(add_row_bias<T>(a.row_bias, v[e], col), add_row_bias<T>(a.row_bias, v[e + 1], col));
                    const int r = 8 * (e >> 2) + (e & 3);
                    if (row0 + r < M) out[(int64_t)r * N] = (uint16_t)pair;
                    if (row0 + r + 1 < M) out[(int64_t)(r + 1) * N] = (uint16_t)(pair >> 16);
                }
            }
        }
    }
}

template <typename T, int BITS, int FP4, bool EXACT, int TI>
int32_t run_tile(ProductArgs a, const splits::Plan &p, void *workspace, hipStream_t s) {
    using S = Shape<BITS, TI>;
    auto kernel = qmk_kernel<T, BITS, FP4, EXACT, TI>;
    static std::atomic<bool> configured{false};
    if (!configured.load()) {
        NVQ_HIP_TRY(hipFuncSetAttribute(reinterpret_cast<const void *>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, S::kLdsBytes));
        configured.store(true);
    }
    a.k_splits = workspace != nullptr ? p.splits : 1;
    a.k_split_steps = (int)p.per_split / (kWin / splits::kQmmStep);  // (splits are whole windows)
    a.partials = a.k_splits > 1 ? static_cast<float *>(workspace) : nullptr;
    const dim3 grid((unsigned)((a.n + kCols - 1) / kCols), (unsigned)((a.m + S::kRows - 1) / S::kRows), (unsigned)(a.batch > 1 ? a.batch : a.k_splits));
    hipLaunchKernelGGL(kernel, grid, dim3(kThreads), S::kLdsBytes, s, a);
    NVQ_LAUNCH_CHECK("qmk");
    return a.k_splits > 1 ? qmm::run_reduce<T>(a, s) : NVQ_OK;
}

template <typename T, int BITS, int FP4, bool EXACT>
int32_t run(const ProductArgs &a, const splits::Plan &p, void *workspace, hipStream_t s) {
    return p.tile == splits::kQmk64 ? run_tile<T, BITS, FP4, EXACT, 2>(a, p, workspace, s) : run_tile<T, BITS, FP4, EXACT, 4>(a, p, workspace, s);
}

template <int BITS, int FP4>
int32_t run_dtype(const ProductArgs &a, const splits::Plan &p, void *workspace, hipStream_t s) {
    if constexpr (FP4 == kAffine)
        if (a.exact_weights) return a.dtype == NVQ_BF16 ? run<bf16_t, BITS, FP4, true>(a, p, workspace, s) : run<f16_t, BITS, FP4, true>(a, p, workspace, s);
    return a.dtype == NVQ_BF16 ? run<bf16_t, BITS, FP4, false>(a, p, workspace, s) : run<f16_t, BITS, FP4, false>(a, p, workspace, s);
}

}  // namespace qmk

// Affine products of few rows and a short K before a bias sum in qmm_kernel's order, as they always did.  The bias is added to the rounded
// product, so that one that nearly cancels it shows that rounding many times over: one of 536640 outputs of 3 bits W[8256,896] at 65
// rows whose product lies 1e-7 of itself beside a rounding boundary falls on either side by the order, here on the one nearer to
// float64, and with the gate and up projections fused into one product on the other.  15 to 16.6 us there, 10.3 to 11.5 here.
inline bool keeps_order(const ProductArgs &a) {
    return a.row_bias != nullptr && a.mode == NVQ_AFFINE && !a.exact_weights && a.m <= 80 && a.k < 1100;
}

// The tiled products of a code width: the plan's kernel.  Products that the dense kernel takes where there is a workspace for it have the
// tile that sums in its order here, K whole, which needs no workspace either.
template <int BITS, int FP4>
int32_t run_tiled(const ProductArgs &a, void *workspace, hipStream_t s) {
    splits::Plan p = qmm_plan_of(a);
    if constexpr (FP4 == qmf::kAffine)
        if (qmm_dense_takes(a) || keeps_order(a)) p = splits::Plan{1, p.units, p.units, 0.0, splits::kSmall};
    if (const char *fault = splits::qmm_plan_fault(p, qmm::split_product(a)))
        return fail(NVQ_BACKEND, "quantized_matmul: the tiled plan has %s (K = %lld in %d parts of %lld steps)", fault, (long long)a.k, p.splits, (long long)p.per_split);
    return p.tile == splits::kBig || p.tile == splits::kSmall ? qmm::run_dtype<BITS, FP4>(a, p, workspace, s) : qmk::run_dtype<BITS, FP4>(a, p, workspace, s);
}

}  // namespace nvq
