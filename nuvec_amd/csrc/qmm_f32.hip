// float32 products of two rows and more on the bfloat16 matrix instruction: y[M,N] = x[M,K] . dequantize(w[N,K])^T for x, scales
// and biases in float32 (the reference instantiates its tiled kernels for float at every width: quantized.metal:40-70,
// fp_quantized.metal:105-107), affine codes of every width, MXFP4, MXFP8 and NVFP4.
//
// v_mfma_f32_16x16x32_bf16 multiplies sixteen times as much a cycle as the float32 instruction and its products are exact, so
// no precision is given up for it:
//   * a code is an exact bfloat16 (integers up to 255, E2M1, E4M3; NVFP4's code times its E4M3 scale has six bits);
//   * x, times 2^26, is the exact sum of three bfloat16 terms of eight bits each, cut off toward zero;
//   * a group's sum P of x times code is formed from the smallest terms up in float32, then y += scale P + bias X with the
//     group's sum X of x.  The biases' part is a product of its own, over groups, on the float32 instruction.
// A weight's own two roundings (crates/nuvec-core/src/kernels.rs:835-859, 992-998), which the CPU's product keeps, are not made.
// What the split of x does not hold, an infinity or a magnitude whose sums of codes leave float32, comes out of it as no finite
// number: a wavefront with such an output multiplies its tiles again, on the float32 instruction.  2^26 makes the
// last term of the least float32, 2^-149, a normal operand (without it magnitudes below 2^-109 lose bits, near 2^-120 most of them).
//
// A block of four wavefronts owns 16 MT rows of x and 64 NT weight rows (16 NT a wavefront) and walks its share of K in steps
// of 64.  x goes through registers, where it is split and its groups' sums are formed, into one of two LDS stages, a step ahead;
// one barrier a step.  Codes come a window ahead in chunks of 16 bytes that consecutive lanes bring, and reach the operand
// layout through a wavefront's own piece of LDS.  Scales and biases come once a span of 256 values, a lane its quarter's.
// Few tiles: K is split over the grid, and qmm_f32_reduce_kernel adds the parts.
//
// What bounds it: a step's vector instructions, two of three for the split of x (a step of 48 rows and 64 weight rows takes 210
// beside 23 matrix instructions, 0.65 us a compute unit; two blocks on one gain a tenth).  Every wavefront reading the
// operands of both halves of a step at once, ahead of the next step's split, gave 0.1 us a step; codes and scales brought
// by each lane for itself, straight in the operand layout, with no LDS and no barrier, was slower by half (16 lines a
// load: W[14336,4096] at 16 rows 28 to 41 us against 20).
#include "qmv_common.h"

#include <math.h>

namespace nvq {
namespace {

using qmf::static_for;

constexpr int kWaves = 4, kThreads = 64 * kWaves;
constexpr int kTile = 16;   // rows of x, weight rows of a matrix instruction
constexpr int kStep = 64;   // values of K between two barriers
constexpr int kSpan = 256;  // values of K of which a lane brings scales and biases; a split of K holds whole ones
constexpr float kLift = 67108864.0f;  // 2^26

template <int BITS, int MODE, int MT, int NT>
struct Shape {
    static constexpr int kRows = kTile * MT, kCols = kTile * NT * kWaves;
    static constexpr int kWindow = BITS <= 4 ? 256 : 128;        // values of K in a window of codes
    static constexpr int kChunks = kWindow * BITS / 128;         // of 16 bytes, of a weight row in a window
    static constexpr int kLoads = (kTile * NT * kChunks + 63) / 64;  // of a lane and window
    static constexpr int kCodeRow = kWindow * BITS / 32 + 4;     // dwords between two weight rows of a window in LDS
    static constexpr int kTermBytes = kRows * kStep * 2, kStageBytes = 3 * kTermBytes;
    static constexpr int kCodeBytes = kTile * NT * kCodeRow * 4;  // of a wavefront
    static constexpr int kSumBytes = kRows * 8 * 4;               // X of a span: eight blocks of 32 or four of 64 a row
    static constexpr int kLds = 2 * kStageBytes + kWaves * kCodeBytes + 2 * kSumBytes;
    static constexpr int kAhead = MT * NT == 8 ? 1 : 2;           // steps of x in registers
};

// Lane i takes the value of lane i ^ 1 (0xB1), i ^ 2 (0x4E), of the mirrored one of its eight (0x141) or sixteen (0x140).
template <int CTRL> __device__ __forceinline__ float lane_swap(float v) {
    return __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, v), CTRL, 0xF, 0xF, true));
}
__device__ __forceinline__ float from_lane(float v, int lane) {
    return __builtin_bit_cast(float, __builtin_amdgcn_ds_bpermute(4 * lane, __builtin_bit_cast(int, v)));
}
__device__ __forceinline__ uint32_t from_lane(uint32_t v, int lane) { return (uint32_t)__builtin_amdgcn_ds_bpermute(4 * lane, (int)v); }

// The high halves of two words: `lo` in the low half.
__device__ __forceinline__ uint32_t high_halves(uint32_t lo, uint32_t hi) { return __builtin_amdgcn_perm(hi, lo, 0x07060302u); }

// Eight codes (in the low 8 BITS bits) as bfloat16, exactly.  Affine codes are taken from the middle of their range, c - 2^(BITS-1)
// (one bit: c - 1/2), times code_factor().
template <int BITS> constexpr float code_factor() { return BITS == 4 ? 16.0f : BITS == 1 ? 2.0f : 1.0f; }
template <int BITS, int MODE>
__device__ __forceinline__ uint4 code_operand(uint64_t codes, float scale) {
    typedef qmf::Ops<bf16_t> Bf;
    uint4 o;
    const uint32_t lo = (uint32_t)codes;
    if constexpr (MODE == NVQ_MXFP4) {
        o.x = Bf::fp4_pair<0>(lo, 1.0f), o.y = Bf::fp4_pair<1>(lo, 1.0f), o.z = Bf::fp4_pair<2>(lo, 1.0f), o.w = Bf::fp4_pair<3>(lo, 1.0f);
    } else if constexpr (MODE == NVQ_NVFP4) {
        o.x = qmf::fp4_pair_times<bf16_t, 0>(lo, scale), o.y = qmf::fp4_pair_times<bf16_t, 1>(lo, scale);
        o.z = qmf::fp4_pair_times<bf16_t, 2>(lo, scale), o.w = qmf::fp4_pair_times<bf16_t, 3>(lo, scale);
    } else if constexpr (MODE == NVQ_MXFP8) {
        const uint32_t hi = (uint32_t)(codes >> 32);
        o.x = Bf::fp8_pair<false>(lo, 1.0f), o.y = Bf::fp8_pair<true>(lo, 1.0f), o.z = Bf::fp8_pair<false>(hi, 1.0f), o.w = Bf::fp8_pair<true>(hi, 1.0f);
    } else {
        // with its top bit turned a code is c - 2^(BITS-1) in two's complement (one bit: from there to twice c - 1/2)
        constexpr uint64_t tops = 0x8080808080808080ull;
        uint32_t f[8];
        if constexpr (BITS == 4) {  // sixteen times it, a byte each
            const uint32_t even = qmf::opaque(((lo << 4) & 0xF0F0F0F0u) ^ 0x80808080u), odd = qmf::opaque((lo & 0xF0F0F0F0u) ^ 0x80808080u);
#pragma unroll
            for (int j = 0; j < 4; j++) f[2 * j] = f2u((float)(int8_t)(even >> (8 * j))), f[2 * j + 1] = f2u((float)(int8_t)(odd >> (8 * j)));
        } else if constexpr (BITS == 8) {
            const uint64_t v = codes ^ tops;
            const uint32_t first = qmf::opaque((uint32_t)v), second = qmf::opaque((uint32_t)(v >> 32));
#pragma unroll
            for (int j = 0; j < 4; j++) f[j] = f2u((float)(int8_t)(first >> (8 * j))), f[4 + j] = f2u((float)(int8_t)(second >> (8 * j)));
        } else {
#pragma unroll
            for (int j = 0; j < 8; j++) {
                const int32_t c = (int32_t)((uint32_t)(codes >> (BITS * j)) << (32 - BITS));
                const int32_t v = (c ^ (int32_t)0x80000000) >> (32 - BITS);
                f[j] = f2u((float)(BITS == 1 ? 2 * v + 1 : v));
            }
        }
        o.x = high_halves(f[0], f[1]), o.y = high_halves(f[2], f[3]), o.z = high_halves(f[4], f[5]), o.w = high_halves(f[6], f[7]);
    }
    return o;
}

// Four weights from value k on (a multiple of four) of weight row `row`, as the CPU dequantizes them: two roundings.
template <int BITS, int MODE>
__device__ __forceinline__ floatx4_t plain_weights(const ProductArgs &a, int64_t row, int k, int gshift, float factor) {
    const int K = (int)a.k;
    const int64_t at = (int64_t)k * BITS;
    const uint32_t *word = (const uint32_t *)a.w + row * (K / 32 * BITS) + at / 32;
    const int bit = (int)(at % 32);
    uint64_t codes = word[0];
    if (bit + 4 * BITS > 32) codes |= (uint64_t)word[1] << 32;  // (a row ends with a dword)
    codes >>= bit;
    const int64_t g = row * (K >> gshift) + (k >> gshift);
    float s, b = 0.0f;
    if constexpr (MODE == NVQ_AFFINE) {
        s = ((const float *)a.scales)[g], b = ((const float *)a.biases)[g];
    } else {
        const uint32_t code = ((const uint8_t *)a.scales)[g];
        s = MODE == NVQ_NVFP4 ? qmf::nvfp4_scale(code, factor) : ftz(e8m0_to_f32(code));
    }
    floatx4_t w;
#pragma unroll
    for (int j = 0; j < 4; j++) {
        const uint32_t c = (uint32_t)(codes >> (BITS * j)) & ((1u << BITS) - 1u);
        w[j] = MODE == NVQ_AFFINE ? (float)c * s + b : (MODE == NVQ_MXFP8 ? e4m3_to_f32(c) : e2m1_to_f32(c)) * s;
    }
    return w;
}

// G32: groups of 32 (affine, MXFP4, MXFP8), whose scale follows every matrix instruction; else blocks of 64, which lie in one group.
template <int BITS, int MODE, int MT, int NT, bool G32>
__global__ void __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(2, MT * NT <= 2 ? 4 : MT * NT == 3 ? 3 : 2))) qmm_f32_kernel(const ProductArgs a) {
    using S = Shape<BITS, MODE, MT, NT>;
    constexpr bool kAffine = MODE == NVQ_AFFINE, kNv = MODE == NVQ_NVFP4;
    constexpr int kBlocks = G32 ? 2 : 1;                 // of a step with a scale of their own
    constexpr int kAhead = S::kAhead;
    constexpr float kMiddle = !kAffine ? 0.0f : BITS == 1 ? 0.5f : (float)(1 << (BITS - 1));
    constexpr int kWindowSteps = S::kWindow / kStep;
    extern __shared__ __attribute__((aligned(16))) unsigned char lds[];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int l = lane & 15, q = lane >> 4;
    const int M = (int)a.m, N = (int)a.n, K = (int)a.k;
    const int gshift = kAffine ? (a.group == 32 ? 5 : a.group == 64 ? 6 : 7) : (kNv ? 4 : 5);
    const int kgroups = K >> gshift, kwords = K / 32 * BITS;
    const int m0 = blockIdx.y * S::kRows, n0 = blockIdx.x * S::kCols + wave * (kTile * NT);
    const int k0 = blockIdx.z * a.k_split_steps * kSpan;
    const int k1 = a.k_splits > 1 && K - k0 > a.k_split_steps * kSpan ? k0 + a.k_split_steps * kSpan : K;
    const int steps = (k1 - k0 + kStep - 1) / kStep;
    unsigned char *code_lds = lds + 2 * S::kStageBytes + wave * S::kCodeBytes;
    float *sum_lds = reinterpret_cast<float *>(lds + 2 * S::kStageBytes + kWaves * S::kCodeBytes);

    // x: a thread brings four values (of a wavefront's 64: four rows) of MT rows of a step; rows past the end repeat the last one and are
    // not stored
    float xs[kAhead][MT][4];  // the next steps', set = step % kAhead
    const int xr = tid >> 4, xc = tid & 15;
    auto load_x = [&](int step, auto set_tag) __attribute__((always_inline)) {
        constexpr int set = decltype(set_tag)::value;
        int k = k0 + step * kStep + 4 * xc;
        k = k < k1 ? k : 0;
#pragma unroll
        for (int m = 0; m < MT; m++) {
            const int row = m0 + kTile * m + xr;
            const float4 v = *reinterpret_cast<const float4 *>((const float *)a.x + (int64_t)(row < M ? row : M - 1) * K + k);
            xs[set][m][0] = v.x, xs[set][m][1] = v.y, xs[set][m][2] = v.z, xs[set][m][3] = v.w;
        }
    };
    // Piece c (eight values) of row r of a term sits at 16-byte place c ^ (r / 2 % 8) of the row: the sixteen rows of an operand read
    // spread over the banks.
    auto store_x = [&](int step, auto set_tag) __attribute__((always_inline)) {
        constexpr int set = decltype(set_tag)::value;
        unsigned char *stage = lds + (step & 1) * S::kStageBytes + xr * (kStep * 2) + (((xc >> 1) ^ (xr >> 1)) * 16) + (xc & 1) * 8;
        // place 4 b + quarter of a row: block `quarter` of 64, or block 2 quarter + b of 32
        float *sums = sum_lds + ((step >> 2) & 1) * (S::kSumBytes / 4) + xr * 8 + (step & 3) + 4 * (xc >> 3);
        if (k0 + (step + 1) * kStep > k1) {  // the last step may be a half
            const bool inside = k0 + step * kStep + 4 * xc < k1;
#pragma unroll
            for (int m = 0; m < MT; m++)
#pragma unroll
                for (int j = 0; j < 4; j++) xs[set][m][j] = inside ? xs[set][m][j] : 0.0f;
        }
#pragma unroll
        for (int m = 0; m < MT; m++) {
            float (&r)[4] = xs[set][m];
#pragma unroll
            for (int j = 0; j < 4; j++) r[j] *= kLift;
            if constexpr (kAffine) {
                float sum = (r[0] + r[1]) + (r[2] + r[3]);
                sum += lane_swap<0xB1>(sum);
                sum += lane_swap<0x4E>(sum);
                sum += lane_swap<0x141>(sum);
                if constexpr (!G32) sum += lane_swap<0x140>(sum);
                if ((xc & (G32 ? 7 : 15)) == 0) sums[kTile * m * 8] = sum;
            }
#pragma unroll
            for (int t = 0; t < 3; t++) {
                uint2 o;
                o.x = high_halves(f2u(r[0]), f2u(r[1])), o.y = high_halves(f2u(r[2]), f2u(r[3]));
                *reinterpret_cast<uint2 *>(stage + t * S::kTermBytes + kTile * m * (kStep * 2)) = o;
#pragma unroll
                for (int j = 0; j < 4; j++) r[j] -= u2f(f2u(r[j]) & 0xFFFF0000u);
            }
        }
    };

    // Codes: the tiles' rows of a window, in order, are cut into chunks of 16 bytes that consecutive lanes bring (rows past the end repeat
    // the last one).  Where K ends inside a chunk the 16 bytes up to its end are brought and moved into place; past the end of K come a
    // row's first bytes, zeroed where a code could be a NaN.
    uint4 cw[S::kLoads];
    auto chunk_of = [&](int i) { const int c = i * 64 + lane; return c < kTile * NT * S::kChunks ? c : 0; };
    auto load_codes = [&](int k) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < S::kLoads; i++) {
            const int n = n0 + chunk_of(i) / S::kChunks;
            int at = k / 32 * BITS + 4 * (chunk_of(i) % S::kChunks);
            at = at >= kwords ? 0 : at + 4 > kwords ? kwords - 4 : at;
            at = at < 0 ? 0 : at;
            cw[i] = __builtin_bit_cast(uint4, *reinterpret_cast<const qmf::u32x4_a4_t *>((const uint32_t *)a.w + (int64_t)(n < N ? n : N - 1) * kwords + at));
        }
    };
    auto store_codes = [&](int k) __attribute__((always_inline)) {
        if (k + S::kWindow > K) {
#pragma unroll
            for (int i = 0; i < S::kLoads; i++) {
                const int at = k / 32 * BITS + 4 * (chunk_of(i) % S::kChunks), missing = at + 4 - kwords;  // dwords past the end
                uint4 &v = cw[i];
                if (missing >= 4) v = make_uint4(0, 0, 0, 0);
                else if (missing == 3) v = make_uint4(v.w, 0, 0, 0);
                else if (missing == 2) v = make_uint4(v.z, v.w, 0, 0);
                else if (missing == 1) v = make_uint4(v.y, v.z, v.w, 0);
            }
        }
#pragma unroll
        for (int i = 0; i < S::kLoads; i++) {
            const int c = i * 64 + lane;
            if ((i + 1) * 64 <= kTile * NT * S::kChunks || c < kTile * NT * S::kChunks)
                *reinterpret_cast<uint4 *>(code_lds + (c / S::kChunks) * (S::kCodeRow * 4) + (c % S::kChunks) * 16) = cw[i];
        }
        __builtin_amdgcn_wave_barrier();  // (the wavefront's LDS accesses execute in order)
    };
    // The eight codes of this lane for block `b` (of 32) of step `j` of the window.
    auto codes_of = [&](int t, int j, int b) __attribute__((always_inline)) {
        const uint32_t *row = reinterpret_cast<const uint32_t *>(code_lds) + (t * kTile + l) * S::kCodeRow + (2 * j + b) * BITS;
        if constexpr (BITS == 4) return (uint64_t)row[q];
        else if constexpr (BITS == 8) return *reinterpret_cast<const uint64_t *>(row + 2 * q);
        else {
            const int first = q * BITS / 4, bit = 8 * (q * BITS % 4);
            uint64_t v = row[first];
            if constexpr (BITS > 2) v |= (uint64_t)row[first + 1 < BITS ? first + 1 : BITS - 1] << 32;
            return v >> bit;
        }
    };

    // Scales and biases of a span: lane (q, l) brings those of step q of the span for weight row l of each tile.
    float sc[NT][kBlocks], bi[NT][kBlocks], sc_next[NT][kBlocks], bi_next[NT][kBlocks];
    uint32_t sw[NT];
    uint8_t sw_next[NT][4];
    auto load_scales = [&](int k) __attribute__((always_inline)) {
#pragma unroll
        for (int t = 0; t < NT; t++) {
            const int n = n0 + kTile * t + l;
            const int64_t row = (int64_t)(n < N ? n : N - 1) * kgroups;
#pragma unroll
            for (int b = 0; b < (kNv ? 4 : kBlocks); b++) {
                const int at = k + q * kStep + b * (kNv ? 16 : 32);
                const int64_t g = row + (at < k1 ? at >> gshift : 0);
                if constexpr (kAffine) sc_next[t][b] = ((const float *)a.scales)[g], bi_next[t][b] = ((const float *)a.biases)[g];
                else sw_next[t][b] = ((const uint8_t *)a.scales)[g];
            }
        }
    };
    // (the middle of the codes' range goes to the bias)
    auto take_scales = [&](int k) __attribute__((always_inline)) {
#pragma unroll
        for (int t = 0; t < NT; t++) {
            if constexpr (kAffine) {
#pragma unroll
                for (int b = 0; b < kBlocks; b++) {
                    const bool inside = k + q * kStep + b * 32 < k1;
                    sc[t][b] = !inside ? 0.0f : sc_next[t][b] * (1.0f / code_factor<BITS>());
                    bi[t][b] = !inside ? 0.0f : __builtin_fmaf(sc_next[t][b], kMiddle, bi_next[t][b]);
                }
            } else {
                sw[t] = 0;
#pragma unroll
                for (int b = 0; b < (kNv ? 4 : 2); b++) sw[t] |= (uint32_t)sw_next[t][b] << (8 * b);
            }
        }
    };

    floatx4_t acc[MT][NT];
#pragma unroll
    for (int m = 0; m < MT; m++)
#pragma unroll
        for (int t = 0; t < NT; t++) acc[m][t] = floatx4_t{0.0f, 0.0f, 0.0f, 0.0f};

    // Every request is made on every path, past the end for something that is not used, and what has come is touched where it is used
    // alone: a wait for one load would be a wait for all.
    load_codes(k0);
    load_scales(k0);
    static_for<kAhead>([&](auto i) { load_x(i, i); });
    store_x(0, std::integral_constant<int, 0>{});
    load_x(kAhead, std::integral_constant<int, 0>{});
    __syncthreads();
    for (int at = 0; at < steps; at += 4) {  // a span
        take_scales(k0 + at * kStep);
        static_for<4>([&](auto j_tag) {
            constexpr int j = decltype(j_tag)::value;
            const int step = at + j;
            if constexpr (j % kWindowSteps == 0) {
                store_codes(k0 + step * kStep);
                load_codes(k0 + (step + kWindowSteps) * kStep);
            }
            if constexpr (j == 0) load_scales(k0 + (step + 4) * kStep);
            // The operands of the step's first half are read, then the next step's x is split while they come.
            const unsigned char *stage = lds + (step & 1) * S::kStageBytes;
            uint64_t codes[2][NT];
            uint4 xo[2][3][MT];
            auto read_x = [&](int b) __attribute__((always_inline)) {
#pragma unroll
                for (int term = 0; term < 3; term++)
#pragma unroll
                    for (int m = 0; m < MT; m++) {
                        const int row = kTile * m + l;
                        xo[b][term][m] = *reinterpret_cast<const uint4 *>(stage + term * S::kTermBytes + row * (kStep * 2) + (((4 * b + q) ^ ((row >> 1) & 7)) * 16));
                    }
            };
#pragma unroll
            for (int b = 0; b < 2; b++)
#pragma unroll
                for (int t = 0; t < NT; t++) codes[b][t] = codes_of(t, j % kWindowSteps, b);
            read_x(0);
            float scale[NT][kBlocks];
            uint32_t word[NT];
#pragma unroll
            for (int t = 0; t < NT; t++) {
                if constexpr (!kAffine) word[t] = from_lane(sw[t], l + 16 * j);
#pragma unroll
                for (int b = 0; b < kBlocks; b++) scale[t][b] = kAffine ? from_lane(sc[t][b], l + 16 * j) : 1.0f;
            }
            __builtin_amdgcn_sched_barrier(0);
            constexpr std::integral_constant<int, (j + 1) % kAhead> set;
            store_x(step + 1, set);
            load_x(step + 1 + kAhead, set);
            uint4 w[2][NT];
#pragma unroll
            for (int t = 0; t < NT; t++) {
                if constexpr (!kAffine && !kNv) {
#pragma unroll
                    for (int b = 0; b < 2; b++) {
                        const uint32_t code = (word[t] >> (8 * b)) & 255u;
                        scale[t][b] = code == 255u ? u2f(0x7FC00000u) : ftz(e8m0_to_f32(code));
                    }
                }
                w[0][t] = code_operand<BITS, MODE>(codes[0][t], kNv ? e4m3_to_f32((word[t] >> (8 * (q >> 1))) & 255u) : 1.0f);
            }
            read_x(1);
            __builtin_amdgcn_sched_barrier(0);
            if (step < steps) {
                floatx4_t p[MT][NT];
                auto multiply = [&](auto b_tag) __attribute__((always_inline)) {
                    constexpr int b = decltype(b_tag)::value;
                    if (G32 || b == 0)
#pragma unroll
                        for (int m = 0; m < MT; m++)
#pragma unroll
                            for (int t = 0; t < NT; t++) p[m][t] = floatx4_t{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
                    for (int term = 2; term >= 0; term--)
#pragma unroll
                        for (int m = 0; m < MT; m++)
#pragma unroll
                            for (int t = 0; t < NT; t++) p[m][t] = Mfma16<bf16_t>::run(xo[b][term][m], w[b][t], p[m][t]);
                    if (b == 0)
#pragma unroll
                        for (int t = 0; t < NT; t++)
                            w[1][t] = code_operand<BITS, MODE>(codes[1][t], kNv ? e4m3_to_f32((word[t] >> (16 + 8 * (q >> 1))) & 255u) : 1.0f);
                    if (G32 || b == 1)
#pragma unroll
                        for (int t = 0; t < NT; t++)
#pragma unroll
                            for (int m = 0; m < MT; m++)
#pragma unroll
                                for (int e = 0; e < 4; e++) acc[m][t][e] = __builtin_fmaf(scale[t][G32 ? b : 0], p[m][t][e], acc[m][t][e]);
                };
                multiply(std::integral_constant<int, 0>{});
                multiply(std::integral_constant<int, 1>{});
            }
            if constexpr (kAffine && j == 3) {  // the span's biases: y += sum over blocks of X[row, block] bias[weight row, block]
                const float *sums = sum_lds + ((step >> 2) & 1) * (S::kSumBytes / 4);
#pragma unroll
                for (int b = 0; b < kBlocks; b++)
#pragma unroll
                    for (int m = 0; m < MT; m++) {
                        const float x = sums[(kTile * m + l) * 8 + 4 * b + q];
#pragma unroll
                        for (int t = 0; t < NT; t++) acc[m][t] = __builtin_amdgcn_mfma_f32_16x16x4f32(x, bi[t][b], acc[m][t], 0, 0, 0);
                    }
            }
            __syncthreads();
        });
    }

    // (the lane's number anew: kept through the loop for these addresses it cost registers, in some shapes a wavefront a SIMD)
    const int end_lane = __builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0u)), el = end_lane & 15, eq = end_lane >> 4;
    const float factor = kNv ? qmf::nvfp4_factor(a, 0) : 1.0f;
    float *y = a.k_splits > 1 ? a.partials + (int64_t)blockIdx.z * M * N : (float *)a.y;
    bool plain = false;
#pragma unroll
    for (int m = 0; m < MT; m++)
#pragma unroll
        for (int t = 0; t < NT; t++)
#pragma unroll
            for (int e = 0; e < 4; e++) {
                if (kNv) acc[m][t][e] *= factor;
                acc[m][t][e] *= 1.0f / kLift;
                plain |= !(fabsf(acc[m][t][e]) < INFINITY);
            }
    // Outputs that are no finite number: the wavefront's tiles again from whole values of x and the CPU's weights on the float32
    // instruction, lane (q, l) with values 4 q .. of sixteen of row l; those outputs alone take what comes.
    if (__any(plain)) {
        floatx4_t again[MT][NT];
#pragma unroll
        for (int m = 0; m < MT; m++)
#pragma unroll
            for (int t = 0; t < NT; t++) again[m][t] = floatx4_t{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll 2
        for (int from = k0; from < k1; from += 16) {
            const int k = from + 4 * eq;
            floatx4_t xv[MT], wv[NT];
#pragma unroll
            for (int m = 0; m < MT; m++) {
                const int row = m0 + kTile * m + el;
                xv[m] = *reinterpret_cast<const floatx4_t *>((const float *)a.x + (int64_t)(row < M ? row : M - 1) * K + k);
            }
#pragma unroll
            for (int t = 0; t < NT; t++) {
                const int n = n0 + kTile * t + el;
                wv[t] = plain_weights<BITS, MODE>(a, n < N ? n : N - 1, k, gshift, factor);
            }
#pragma unroll
            for (int j = 0; j < 4; j++)
#pragma unroll
                for (int m = 0; m < MT; m++)
#pragma unroll
                    for (int t = 0; t < NT; t++) again[m][t] = __builtin_amdgcn_mfma_f32_16x16x4f32(xv[m][j], wv[t][j], again[m][t], 0, 0, 0);
        }
#pragma unroll
        for (int m = 0; m < MT; m++)
#pragma unroll
            for (int t = 0; t < NT; t++)
#pragma unroll
                for (int e = 0; e < 4; e++) acc[m][t][e] = fabsf(acc[m][t][e]) < INFINITY ? acc[m][t][e] : again[m][t][e];
    }
    // Accumulator element e of lane (q, l): row 4 q + e of x, weight row l.
#pragma unroll
    for (int m = 0; m < MT; m++)
#pragma unroll
        for (int t = 0; t < NT; t++)
#pragma unroll
            for (int e = 0; e < 4; e++) {
                const int row = m0 + kTile * m + 4 * eq + e, col = n0 + kTile * t + el;
                if (row < M && col < N) y[(int64_t)row * N + col] = a.k_splits > 1 ? acc[m][t][e] : add_row_bias<float>(a.row_bias, acc[m][t][e], col);
            }
}

// The parts of a split K, eight under way at a time and added by pairs.
__global__ void __launch_bounds__(256) qmm_f32_reduce_kernel(const float *__restrict__ partials, float *__restrict__ y, int splits, int64_t total,
                                                             const void *row_bias, int64_t n) {
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= total) return;
    float sum = 0.0f;
    for (int s = 0; s < splits; s += 8) {
        float v[8];
#pragma unroll
        for (int u = 0; u < 8; u++) v[u] = partials[(int64_t)(s + u < splits ? s + u : s) * total + i];
#pragma unroll
        for (int u = 0; u < 8; u++) v[u] = s + u < splits ? v[u] : 0.0f;
        sum += ((v[0] + v[1]) + (v[2] + v[3])) + ((v[4] + v[5]) + (v[6] + v[7]));
    }
    y[i] = add_row_bias<float>(row_bias, sum, i % n);
}

struct Plan {
    int mt, nt, splits, spans;  // tiles of rows of x a block, of weight rows a wavefront; spans of K a split
    double us;                  // estimated
};

// The tiles of weight rows and the split of K with the least estimated time.  Fitted (14 % off on average) to 3700 timings of 552
// products of 2 to 512 rows, twelve weight shapes from W[600,2496] to W[33000,512] and W[4096,14336], 4 and 8 bits, MXFP8 and NVFP4: a
// step costs a compute unit 0.12 + 0.17 us per tile of rows at 64 weight rows a block, 0.25 + 0.28 at 128, whether its blocks run one
// after the other or side by side; choosing by it is 4 % above always taking the fastest.  The parts fit the library's own scratch.
Plan plan_of(const ProductArgs &a) {
    Plan best{};
    const int64_t tiles = (a.m + kTile - 1) / kTile, passes = (tiles + 3) / 4, spans = (a.k + kSpan - 1) / kSpan, steps = (a.k + kStep - 1) / kStep;
    const int mt = (int)((tiles + passes - 1) / passes);
    const double cus = fmax(1.0, (double)compute_units()), outputs = (double)a.m * (double)a.n;
    for (int nt = 1; nt <= 2; nt++)
        for (int64_t want = 1; want <= 16 && want <= spans; want++) {
            const int64_t per = (spans + want - 1) / want, splits = (spans + per - 1) / per;
            if (splits != want || (splits > 1 && (double)splits * outputs * 4.0 > (double)NVQ_STATIC_SCRATCH_BYTES)) continue;
            const double load = (double)(passes * ((a.n + 64 * nt - 1) / (64 * nt)) * splits) / cus;
            const double step_us = nt == 1 ? 0.12 + 0.17 * mt : 0.25 + 0.28 * mt;
            const double us = 5.3 + (double)(4 * per < steps ? 4 * per : steps) * step_us * fmax(1.0, 0.25 * ceil(load) + 0.75 * load) +
                              (splits > 1 ? 1.3 + 1.1e-6 * (double)splits * outputs : 0.0);
            if (best.nt == 0 || us < best.us) best = Plan{mt, nt, (int)splits, (int)per, us};
        }
    return best;
}

template <int BITS, int MODE, int MT, int NT, bool G32>
int32_t run_shape(const ProductArgs &a, hipStream_t s) {
    constexpr int kLds = Shape<BITS, MODE, MT, NT>::kLds;
    auto kernel = qmm_f32_kernel<BITS, MODE, MT, NT, G32>;
    static std::atomic<bool> configured{false};
    if (kLds > 64 * 1024 && !configured.load()) {
        NVQ_HIP_TRY(hipFuncSetAttribute(reinterpret_cast<const void *>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, kLds));
        configured.store(true);
    }
    const dim3 grid((unsigned)((a.n + 64 * NT - 1) / (64 * NT)), (unsigned)((a.m + kTile * MT - 1) / (kTile * MT)), (unsigned)a.k_splits);
    hipLaunchKernelGGL(kernel, grid, dim3(kThreads), kLds, s, a);
    NVQ_LAUNCH_CHECK("qmm_f32");
    return NVQ_OK;
}

template <int BITS, int MODE, int NT, bool G32>
int32_t run_rows(const ProductArgs &a, int mt, hipStream_t s) {
    switch (mt) {
    case 1: return run_shape<BITS, MODE, 1, NT, G32>(a, s);
    case 2: return run_shape<BITS, MODE, 2, NT, G32>(a, s);
    case 3: return run_shape<BITS, MODE, 3, NT, G32>(a, s);
    default: return run_shape<BITS, MODE, 4, NT, G32>(a, s);
    }
}

template <int BITS, int MODE = NVQ_AFFINE>
int32_t run(const ProductArgs &a, const Plan &p, hipStream_t s) {
    if constexpr (MODE == NVQ_AFFINE) {
        if (a.group != 32) return p.nt == 1 ? run_rows<BITS, MODE, 1, false>(a, p.mt, s) : run_rows<BITS, MODE, 2, false>(a, p.mt, s);
    }
    constexpr bool kG32 = MODE != NVQ_NVFP4;
    return p.nt == 1 ? run_rows<BITS, MODE, 1, kG32>(a, p.mt, s) : run_rows<BITS, MODE, 2, kG32>(a, p.mt, s);
}

}  // namespace

// What the kernel takes: one product (no batch, no gathered pairs, no gated epilogue, not row-exact) of float32 x against weights
// stored [N, K], K in whole blocks of 32.
static bool qmm_f32_supported(const ProductArgs &a) {
    if (a.dtype != NVQ_F32 || a.row_exact || a.batch != 1 || a.batch_ndim != 0 || a.rhs != nullptr || a.lhs != nullptr || a.glu != 0) return false;
    if (a.m < 2 || a.k < 32 || a.k % 32 != 0 || (a.mode == NVQ_AFFINE && a.group != 32 && a.group != 64 && a.group != 128)) return false;
    if (a.k / 32 * a.bits < 4) return false;  // (a chunk of codes lies inside a row)
    return (a.m + 15) / 16 <= 65535 && a.n <= 0x7FFFFFFF / 64 && a.k <= 1 << 26 && (uintptr_t)a.x % 16 == 0;
}

// Where it is estimated faster than the vector kernel, which walks the weights once per four rows of x: 4 us and a pass of four rows at
// 1 us per 2.1 M weights, K counted in its steps of 2048 values (E2M1 codes 2.5 times that).  Timed on the 552 products of plan_of it
// takes 0.28 of the time of what served them before, the vector kernel and two on v_mfma_f32_16x16x4_f32 and 32x32x2 (4 bits, us:
// W[4096,4096] at 33 / 64 / 128 / 512 rows 35 / 45 / 87 / 178 -> 17 / 22 / 30 / 70, W[14336,4096] at 16 rows 76 -> 20, W[704,5376] at
// 274 rows 134 -> 23), and its error against float64 is lower (W[4096,4096] at 33 rows 2.9e-7 -> 1.0e-7, 2.9e-7 -> 1.0e-7 for NVFP4).
bool qmm_f32_faster(const ProductArgs &a, double margin) {
    if (!qmm_f32_supported(a)) return false;
    const bool e2m1 = a.mode == NVQ_MXFP4 || a.mode == NVQ_NVFP4;
    const double k_steps = (double)((a.k + 2047) / 2048) * 2048.0;
    return plan_of(a).us < margin * (4.0 + (e2m1 ? 2.52 : 1.05) * (double)((a.m + 3) / 4) * (double)a.n * k_steps / 2.2e6);
}

// Whether the product's route is this kernel's name.  A few rows of affine and E4M3 codes (of 1024 values and more up to 4, of whole steps
// of 2048 up to 8, against up to 2^24 weights up to 32), four rows of MXFP4 up to 2^24 weights and more than 128 rows of K off whole
// steps of 64 keep the vector kernel's, by which callers that ask for a route know them.
bool qmm_f32_takes(const ProductArgs &a) {
    if (a.k % kStep != 0 && a.m > 128) return false;
    const bool small = a.n * a.k <= 1 << 24, e2m1 = a.mode == NVQ_MXFP4 || a.mode == NVQ_NVFP4;
    if (!e2m1 && (a.k % 2048 == 0 ? a.m <= (small ? 32 : 8) : a.k >= 1024 && a.m <= 4)) return false;
    return !(a.mode == NVQ_MXFP4 && small && a.m <= 4) && qmm_f32_faster(a, 1.0);
}

size_t qmm_f32_workspace_bytes(const ProductArgs &a) {
    const Plan p = plan_of(a);
    return p.splits > 1 ? (size_t)p.splits * (size_t)a.m * (size_t)a.n * sizeof(float) : 0;
}

int32_t launch_qmm_f32(const ProductArgs &args, void *workspace, hipStream_t s) {
    if (!qmm_f32_supported(args)) return fail(NVQ_UNSUPPORTED, "quantized_matmul: the float32 matrix-core kernel does not take this product");
    ProductArgs a = args;
    const Plan p = plan_of(a);
    a.k_splits = workspace != nullptr ? p.splits : 1;
    a.k_split_steps = p.spans;
    a.partials = (float *)workspace;
    int32_t rc;
    if (a.mode == NVQ_MXFP4) rc = run<4, NVQ_MXFP4>(a, p, s);
    else if (a.mode == NVQ_MXFP8) rc = run<8, NVQ_MXFP8>(a, p, s);
    else if (a.mode == NVQ_NVFP4) rc = run<4, NVQ_NVFP4>(a, p, s);
    else switch (a.bits) {
    case 1: rc = run<1>(a, p, s); break;
    case 2: rc = run<2>(a, p, s); break;
    case 3: rc = run<3>(a, p, s); break;
    case 4: rc = run<4>(a, p, s); break;
    case 5: rc = run<5>(a, p, s); break;
    case 6: rc = run<6>(a, p, s); break;
    case 8: rc = run<8>(a, p, s); break;
    default: return fail(NVQ_INVALID_ARGUMENT, "quantized_matmul: %d bits are not supported", a.bits);
    }
    if (rc != NVQ_OK || a.k_splits <= 1) return rc;
    const int64_t total = a.m * a.n;
    hipLaunchKernelGGL(qmm_f32_reduce_kernel, dim3((unsigned)((total + 255) / 256)), dim3(256), 0, s, a.partials, (float *)a.y, a.k_splits, total, a.row_bias, a.n);
    NVQ_LAUNCH_CHECK("qmm_f32_reduce");
    return NVQ_OK;
}

}  // namespace nvq
