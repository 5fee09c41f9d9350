// float32 products of a few rows on the matrix cores: y[M,N] = x[M,K] . dequantize(w[N,K])^T for x, scales and biases in
// float32, on v_mfma_f32_16x16x4_f32.  Weights as in qmm_f32.hip: dequantized in float32 exactly as nuvec's CPU product does
// (reference: crates/nuvec-core/src/kernels.rs:835-859, 992-998), sums in float32 (kernels.rs:1091-1142).
//
// What bounds it is the matrix instruction (256 operations a cycle and compute unit, a sixteenth of bfloat16's), so rows come
// in tiles of 16 and not of 64: 33 rows cost 48.  A wavefront owns 16 weight rows and up to 64 rows of x and walks its share
// of K in windows of 32 values; the wavefronts of a block share K (KW of them a tile) until the chip is full, and their sums
// meet in LDS.  Nothing is staged: lane (quarter q, l) takes values 8 q .. 8 q + 7 of a window of its weight row, which are
// BITS whole bytes of codes, and of its rows of x, 32 bytes each, so that a wavefront's load touches sixteen lines; both
// operands keep that order of K.  Two windows are under way while one is multiplied.  The number of loads a window is what
// it costs beside the matrix instructions: with two runs of four values a lane and four windows under way 33 rows of
// W[4096,4096] took 40 us against 34, two rows of W[62208,512] 50 against 32.
//
// us, vector kernel (a pass over the weights per four rows) or the 64 x 64 tiles -> this one, 4-bit g64: W[4096,4096] at 33 /
// 48 / 96 rows 71 / 94 / 106 -> 34 / 38 / 73, W[4096,14336] at 33 rows 236 -> 114, W[62208,512] at 5 rows 119 -> 34.
#include "nvq_device.h"
#include "nvq_internal.h"
#include "qmf_kernel.h"

#include <math.h>

namespace nvq {
namespace {

using qmf::static_for;

typedef float f32x4_t __attribute__((ext_vector_type(4)));

constexpr int kWaves = 8;
constexpr int kTile = 16;    // weight rows of a wavefront; rows of x of a tile
constexpr int kWindow = 32;  // values of K

// MODE: NVQ_AFFINE, NVQ_MXFP4, NVQ_MXFP8 or NVQ_NVFP4 (BITS is 4 or 8 for the block formats); MT tiles of rows of x.
template <int BITS, int MODE, int MT>
__global__ void __launch_bounds__(64 * kWaves, MT <= 3 ? 4 : 2) qmf_f32_kernel(const ProductArgs a, int kw_shift) {
    constexpr bool kAffine = MODE == NVQ_AFFINE;
    constexpr int kDwords = BITS == 1 || BITS == 2 || BITS == 4 ? 1 : 2;  // that hold a lane's eight codes
    constexpr int kStride = kTile + 1;
    __shared__ float part[kWaves][MT * kTile * kStride];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int l = lane & 15, q = lane >> 4;
    const int M = (int)a.m, N = (int)a.n, K = (int)a.k;
    const int gshift = kAffine ? (a.group == 32 ? 5 : a.group == 64 ? 6 : 7) : (MODE == NVQ_NVFP4 ? 4 : 5);
    const int kgroups = K >> gshift, windows = K / kWindow;
    const int kw = 1 << kw_shift, k_part = wave & (kw - 1);
    const int n0 = (blockIdx.x * (kWaves >> kw_shift) + (wave >> kw_shift)) * kTile, m0 = blockIdx.y * (MT * kTile);

    // (rows past the ends read the last one and are not stored)
    const int n = n0 + l < N ? n0 + l : N - 1;
    const float *xrow[MT];
#pragma unroll
    for (int t = 0; t < MT; t++) xrow[t] = (const float *)a.x + (int64_t)(m0 + kTile * t + l < M ? m0 + kTile * t + l : M - 1) * K + 8 * q;
    const uint32_t *wrow = (const uint32_t *)a.w + (int64_t)n * windows * BITS;
    const int first = q * BITS / 4, bit = 8 * (q * BITS % 4);  // of the codes: dword of a window's BITS, bit in it
    const int second = first + 1 < BITS ? first + 1 : BITS - 1;
    const float *srow = (const float *)a.scales + (int64_t)n * kgroups, *brow = (const float *)a.biases + (int64_t)n * kgroups;
    const uint8_t *crow = (const uint8_t *)a.scales + (int64_t)n * kgroups;  // block formats
    float inv_enc = 1.0f;
    bool scaled = false;
    if constexpr (MODE == NVQ_NVFP4) {
        if (a.global_scale != nullptr) inv_enc = ftz(a.global_scale[0] / (448.0f * 6.0f)), scaled = true;
    }

    struct Window {
        f32x4_t x[MT][2];
        uint32_t c[kDwords];
        float s, b;
        uint32_t code;  // block formats: of the scale
    } win[2];
    auto fetch = [&](int at, Window &o) __attribute__((always_inline)) {
        const int i = at < windows ? at : windows - 1;  // (past the end: read, not used)
#pragma unroll
        for (int t = 0; t < MT; t++)
#pragma unroll
            for (int p = 0; p < 2; p++) o.x[t][p] = *reinterpret_cast<const f32x4_t *>(xrow[t] + i * kWindow + 4 * p);
        o.c[0] = wrow[i * BITS + first];
        if constexpr (kDwords == 2) o.c[1] = wrow[i * BITS + second];
        const int g = (i * kWindow + 8 * q) >> gshift;
        if constexpr (kAffine) o.s = srow[g], o.b = brow[g];
        else o.code = crow[g];
    };
    f32x4_t acc[MT][2];
#pragma unroll
    for (int t = 0; t < MT; t++) acc[t][0] = acc[t][1] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
    auto multiply = [&](const Window &o) __attribute__((always_inline)) {
        uint64_t codes = o.c[0];
        if constexpr (kDwords == 2) codes |= (uint64_t)o.c[1] << 32;
        if constexpr (BITS != 4 && BITS != 8) codes >>= bit;
        float scale = 0.0f;
        if constexpr (kAffine) {
            scale = o.s;
        } else {
            scale = ftz(MODE == NVQ_NVFP4 ? e4m3_to_f32(o.code) : e8m0_to_f32(o.code));
            if (scaled) scale = ftz(scale * inv_enc);
        }
        static_for<8>([&](auto j_tag) {
            constexpr int j = decltype(j_tag)::value;
            const uint32_t c = (uint32_t)(codes >> (BITS * j)) & ((1u << BITS) - 1u);
            float wv;
            if constexpr (kAffine) wv = (float)c * scale + o.b;  // two roundings, as the CPU's weight
            else wv = (MODE == NVQ_MXFP8 ? e4m3_to_f32(c) : e2m1_to_f32(c)) * scale;
#pragma unroll
            for (int t = 0; t < MT; t++) acc[t][j & 1] = __builtin_amdgcn_mfma_f32_16x16x4f32(o.x[t][j >> 2][j & 3], wv, acc[t][j & 1], 0, 0, 0);
        });
    };
    fetch(k_part, win[0]);
    fetch(k_part + kw, win[1]);
    for (int i = k_part; i < windows; i += 2 * kw) {
        multiply(win[0]);
        fetch(i + 2 * kw, win[0]);
        if (i + kw < windows) multiply(win[1]);
        fetch(i + 3 * kw, win[1]);
    }

    // Accumulator element e of lane (q, l): row 4 q + e of x, weight row l.
#pragma unroll
    for (int t = 0; t < MT; t++)
#pragma unroll
        for (int e = 0; e < 4; e++) part[wave][(kTile * t + 4 * q + e) * kStride + l] = acc[t][0][e] + acc[t][1][e];
    __syncthreads();
    float *y = (float *)a.y;
    const int cols = kTile * (kWaves >> kw_shift), block_n0 = blockIdx.x * cols;
    for (int i = tid; i < cols * MT * kTile; i += 64 * kWaves) {
        const int col = i & (cols - 1), row = i / cols, w0 = (col / kTile) << kw_shift;
        float sum = 0.0f;
        for (int k = 0; k < kw; k++) sum += part[w0 + k][row * kStride + col % kTile];
        if (m0 + row < M && block_n0 + col < N) y[(int64_t)(m0 + row) * N + block_n0 + col] = add_row_bias<float>(a.row_bias, sum, block_n0 + col);
    }
}

int64_t row_tiles(const ProductArgs &a) { return (a.m + kTile - 1) / kTile; }
int64_t row_passes(const ProductArgs &a) { return (row_tiles(a) + 3) / 4; }

// Wavefronts of a tile, a power of two: sixteen a compute unit (what the registers let run together) where the tiles alone are fewer.
int tile_waves_shift(const ProductArgs &a) {
    const int64_t tiles = (a.n + kTile - 1) / kTile * row_passes(a);
    int shift = 0;
    while (shift < 3 && (tiles << shift) < 16 * (int64_t)compute_units() && (2 << shift) <= a.k / kWindow) shift++;
    return shift;
}

template <int BITS, int MODE = NVQ_AFFINE>
int32_t run(const ProductArgs &a, hipStream_t s) {
    const int64_t passes = row_passes(a);
    const int shift = tile_waves_shift(a);
    const int64_t cols = kTile * (kWaves >> shift);
    const dim3 grid((unsigned)((a.n + cols - 1) / cols), (unsigned)passes), block(64 * kWaves);
    switch ((row_tiles(a) + passes - 1) / passes) {
    case 1: hipLaunchKernelGGL((qmf_f32_kernel<BITS, MODE, 1>), grid, block, 0, s, a, shift); break;
    case 2: hipLaunchKernelGGL((qmf_f32_kernel<BITS, MODE, 2>), grid, block, 0, s, a, shift); break;
    case 3: hipLaunchKernelGGL((qmf_f32_kernel<BITS, MODE, 3>), grid, block, 0, s, a, shift); break;
    default: hipLaunchKernelGGL((qmf_f32_kernel<BITS, MODE, 4>), grid, block, 0, s, a, shift); break;
    }
    NVQ_LAUNCH_CHECK("qmf_f32");
    return NVQ_OK;
}

}  // namespace

// One product (no batch, no gathered pairs, no gated epilogue, not row-exact) of float32 x against weights stored [N, K], K in
// whole windows.
bool qmf_f32_supported(const ProductArgs &a) {
    if (a.dtype != NVQ_F32 || a.row_exact || a.batch != 1 || a.batch_ndim != 0 || a.rhs != nullptr || a.lhs != nullptr || a.glu != 0) return false;
    return a.k >= kWindow && a.k % kWindow == 0 && row_passes(a) <= 65535 && a.n <= 0x7FFFFFFF / 64;
}

// Where it is estimated faster than the kernel that takes the product otherwise (qmm_f32_takes says which).  All three were timed on
// 2486 products (18 weight shapes from W[2000,1920] to W[100000,1024] and W[4096,14336], 11 formats, 2 to 128 rows, weights from
// memory).  A window costs a tile that a block's eight wavefronts share `window` us and `tile` us per tile of rows, four tiles `four` us
// in all, and a compute unit its blocks one after the other; where they do not divide evenly the time lies between the average and the
// fullest unit's (8.7 to 13 % off on average).  The others' estimates are those of qmm_f32_takes times a factor per kind of code: the
// vector kernel takes E2M1 codes twice as long, E4M3 codes no longer than affine ones, and one pass over the weights for two to
// four rows.  Choosing by them is 0.3 to 0.8 % above always taking the faster kernel; of 3431 products timed with the rule, 945 of them of
// other shapes, 14 take more than 5 % longer than without this kernel, 1.10 x at worst, and all together 0.71 of the time (by one
// factor for all block formats, fitted to eight rows and more, MXFP8 W[1024,8192] at 48 rows took 74 us for 49, W[100000,1024] at 4 rows
// 114 for 86).  Left to the vector kernel, us there / here: W[14336,4096] at 2 rows
// 30 / 59, W[4096,14336] at 7 rows 60 / 75; taken: W[62208,512] at 2 rows 61 / 32, W[33000,544] at 4 rows 36 / 18, MXFP4 W[14336,4096]
// at 5 rows 105 / 47.  Up to 32 rows of matrices up to W[4096,4096] stay on the vector kernel, more than 128 rows on the tiles: the
// kernel was not timed there.
bool qmf_f32_takes(const ProductArgs &a) {
    if (!qmf_f32_supported(a) || a.m < 2 || a.m > 128) return false;
    if (a.m <= 32 && a.n * a.k <= 4096LL * 4096) return false;
    struct Fit { double window, tile, four, vector, tiles; };
    const Fit fit = a.mode == NVQ_MXFP8          ? Fit{0.046, 0.072, 0.346, 1.06, 1.34}
                    : a.mode != NVQ_AFFINE       ? Fit{0.038, 0.059, 0.294, 2.52, 1.50}
                    : a.bits == 3 || a.bits == 8 ? Fit{0.090, 0.064, 0.361, 1.04, 0.92}
                                                 : Fit{0.065, 0.064, 0.336, 1.04, 0.92};
    const double rows = ceil((double)row_tiles(a) / (double)row_passes(a)), units = compute_units();
    const int64_t tiles = kWaves >> tile_waves_shift(a);  // of a block
    const double blocks = (double)((a.n + kTile * tiles - 1) / (kTile * tiles)) * (double)row_passes(a) / units;
    const double shared = fmax(1.0, (0.6 * ceil(blocks) + 0.4 * blocks) * (double)tiles);
    const double here = 2.5 + shared * (double)(a.k / kWindow) * (rows > 3.0 ? fit.four : fit.window + fit.tile * rows);
    if (qmm_f32_takes(a)) {
        const double tiles64 = (double)((a.m + 63) / 64) * (double)((a.n + 63) / 64);
        return here < fit.tiles * (double)(a.k / 64) * fmax(1.64, 1.25 * tiles64 / units);
    }
    const double k_steps = (double)((a.k + 2047) / 2048) * 2048.0;
    return here < fit.vector * (double)((a.m + 3) / 4) * (double)a.n * k_steps / 2.2e6;
}

int32_t launch_qmf_f32(const ProductArgs &a, hipStream_t s) {
    if (!qmf_f32_supported(a)) return fail(NVQ_UNSUPPORTED, "quantized_matmul: the few-row float32 kernel does not take this product");
    if (a.mode == NVQ_MXFP4) return run<4, NVQ_MXFP4>(a, s);
    if (a.mode == NVQ_MXFP8) return run<8, NVQ_MXFP8>(a, s);
    if (a.mode == NVQ_NVFP4) return run<4, NVQ_NVFP4>(a, s);
    switch (a.bits) {
    case 1: return run<1>(a, s);
    case 2: return run<2>(a, s);
    case 3: return run<3>(a, s);
    case 4: return run<4>(a, s);
    case 5: return run<5>(a, s);
    case 6: return run<6>(a, s);
    case 8: return run<8>(a, s);
    default: return fail(NVQ_INVALID_ARGUMENT, "quantized_matmul: %d bits are not supported", a.bits);
    }
}

}  // namespace nvq
