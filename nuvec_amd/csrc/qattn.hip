// Attention of one query row per head over an affine-quantized key / value cache: the counterpart of
// the reference's FastOp::QuantizedAttention kernel (crates/nuvec-core/src/fast.rs:694-718; its fit rule
// crates/nuvec-core/src/fast/imp.rs:3944-3992; launch crates/nuvec-core/src/gpu.rs:4969-5040):
//     out[b, h, :] = softmax(scale * q[b, h, :] . K[b, h / rep]^T [, sink[h]]) . V[b, h / rep]
// with K and V stored packed (codes [B, Hkv, S, D bits / 32], scales and biases [B, Hkv, S, D / group]).  Products and sums
// are float32 and the codes are never rounded (the reference's kernel likewise: "within the float bound of the dequantized
// attention").
//
// The bound is the stream of the cache, read once for all query heads of a key head, as long as turning codes into operands
// costs little: both products run on the matrix cores over the CODES, which bfloat16 holds exactly (8 bits as they are, 3 and
// 4 bits in the mantissa of 8 and 16: one instruction per two codes, the 8 or 16 taken out again by the sums it multiplies;
// in the mantissa of 128 float32 results lost a digit).  The values' sums count codes from the middle of their range, as large
// as the values around their mean, so that the weights' rounding is not multiplied by the range: the operands themselves in
// float32, else by an operand of the offset and the middle alone that goes through the same sums.
// What is not exact in bfloat16, the queries of the wider types and the softmax's weights, goes in as the sum of bfloat16 terms of
// 8 bits each: a float16 query in two, a float32 query and the weights of every type, float32 values, in three (TQ and TP below).
// Errors against float64, weights and sums in float32 on the vector units as they were -> here: float16 2.01e-4 .. 2.10e-4 -> the
// same to four digits (the output's rounding; with two terms of the weights a ten-thousandth more), float32 3.6e-7 .. 5.4e-7 ->
// 1.8e-7 .. 2.8e-7, on the vector kernel below 1.6e-7 .. 2.3e-7.  The third term costs 3 to 4 % (16 x 8 heads x 8192 positions of 4
// bits 51.2 -> 53.4 us).
//
// With few query heads per key head or few positions most of an instruction's columns or of the chip stays empty: those take a
// vector kernel, one query head a block (vector_is_faster).
//
// Groups.  v_mfma_f32_16x16x32 has 16 columns and a key head at most 8 query heads: the columns are (group of D, query head)
// with 16 / groups heads each (eight heads over four groups take two blocks).  The query's operand holds zeros outside
// a column's group, so S^T = K . Q^T separates the groups' partial scores without regard to which codes share an
// instruction, and a lane's 32 codes (16 bytes at 4 bits) are consecutive; scale and bias of a column's group are applied to
// the partial score, the groups of a row are added across lanes.  In O^T = V^T . P^T a column's weights are p times that
// group's scale: a row of D is taken from the columns of its own group, the others are ignored.
//
// Lanes.  Lane (quarter q, l) holds in S^T column l of keys 4 q .. + 3 of two tiles of 16 keys: they are the eight keys of its
// operand P^T (the contraction's order is free), and of V it loads D / 16 codes, l's slot of the row, of the same eight keys.
// No value crosses lanes but the groups' sums, and maxima when they grow.
#include "attention_merge.h"
#include "nvq_device.h"
#include "nvq_internal.h"
#include "qmf_kernel.h"

namespace nvq {
namespace {

typedef float floatx4_t __attribute__((ext_vector_type(4)));
constexpr int kAttnWaves = 4;
constexpr int kTileKeys = 32;
constexpr float kLog2e = 1.44269504088896340736f;

__device__ __forceinline__ floatx4_t mfma16(uint4 a, uint4 b, floatx4_t c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(qmf::bf16x8_t, a), __builtin_bit_cast(qmf::bf16x8_t, b), c, 0, 0, 0);
}

// A value from any address, in as few loads as it has dwords.
template <typename V>
__device__ __forceinline__ V load_any(const void *p) {
    struct __attribute__((packed)) Raw { V v; };
    return reinterpret_cast<const Raw *>(p)->v;
}

// An operand is kOffset + code.  WIDE: float32.
template <int BITS, bool WIDE> constexpr float kOffset = WIDE ? -(float)(1 << (BITS - 1)) : BITS == 8 ? 0.0f : (float)(1 << BITS);
template <int BITS> constexpr uint32_t kMagic = BITS == 4 ? 0x41804180u : 0x41004100u;  // two of 2^BITS, BITS < 8
// Codes at bit `at` of both halves of a word as 2^BITS + code.  The constants come in registers, a scalar one and a vector one: then the
// mask and the exponent are one instruction (v_and_or_b32, which takes no literal; from constants they were two).
template <int BITS>
struct CodeConstants {
    uint32_t mask = ((1u << BITS) - 1u) * 0x00010001u << (7 - BITS), magic = kMagic<BITS>;
    __device__ __forceinline__ CodeConstants() {
        asm("" : "+s"(mask));
        asm("" : "+v"(magic));
    }
};
template <int BITS>
__device__ __forceinline__ uint32_t two_codes(const CodeConstants<BITS> &c, uint32_t z, int at) {
    constexpr int to = 7 - BITS;  // the code's place in the mantissa
    return ((at >= to ? z >> (at - to) : z << (to - at)) & c.mask) | c.magic;
}

// Two exact bfloat16 values from two floats that bfloat16 holds.
__device__ __forceinline__ uint32_t pack_exact(float lo, float hi) { return __builtin_amdgcn_perm(f2u(hi), f2u(lo), 0x07060302u); }

// Which of eight consecutive codes element j of an operand is.
template <int BITS> constexpr int code_at(int j) { return BITS == 8 ? j : (j >> 1) + 4 * (j & 1); }

// Eight consecutive codes of a row (BITS bytes in the low bits of w0, w1) as an operand, in the order of code_at.
template <int BITS, bool WIDE>
__device__ __forceinline__ uint4 eight_codes(const CodeConstants<BITS> &c, uint32_t w0, uint32_t w1) {
    if constexpr (WIDE) {
        auto at = [&](int j) {
            const int i = code_at<BITS>(j);
            const uint32_t code = BITS == 8 ? (i < 4 ? w0 >> (8 * i) : w1 >> (8 * (i - 4))) & 0xFFu : (w0 >> (BITS * i)) & ((1u << BITS) - 1u);
            return (float)code + kOffset<BITS, true>;
        };
        return make_uint4(pack_exact(at(0), at(1)), pack_exact(at(2), at(3)), pack_exact(at(4), at(5)), pack_exact(at(6), at(7)));
    } else if constexpr (BITS == 8) {
        return make_uint4(pack_exact(qmf::ubyte_to_float<0>(w0), qmf::ubyte_to_float<1>(w0)), pack_exact(qmf::ubyte_to_float<2>(w0), qmf::ubyte_to_float<3>(w0)),
                          pack_exact(qmf::ubyte_to_float<0>(w1), qmf::ubyte_to_float<1>(w1)), pack_exact(qmf::ubyte_to_float<2>(w1), qmf::ubyte_to_float<3>(w1)));
    } else {
        const uint32_t z = BITS == 4 ? w0 : (w0 & 0xFFFu) | ((w0 & 0xFFF000u) << 4);  // code i at bit BITS i, code i + 4 sixteen above
        return make_uint4(two_codes(c, z, 0), two_codes(c, z, BITS), two_codes(c, z, 2 * BITS), two_codes(c, z, 3 * BITS));
    }
}

// Keys of one split of the positions: whole tiles of all wavefronts of a block, so that no tile is shared.
__host__ __device__ inline int attention_split_keys(int64_t positions, int splits) {
    const int64_t per = (positions + splits - 1) / splits;
    return (int)((per + kTileKeys - 1) / kTileKeys * kTileKeys);
}

// A float as a sum of N bfloat16 terms (8 bits each), two floats at a time: term i of both in t[i].
template <int N>
__device__ __forceinline__ void split_pair(float a, float b, uint32_t (&t)[N]) {
#pragma unroll
    for (int i = 0; i < N; i++) {
        t[i] = f32_to_bf16_pair(a, b);
        a -= u2f(t[i] << 16), b -= u2f(t[i] & 0xFFFF0000u);
    }
}

// Blocks on a compute unit.  Three need 168 registers at most: there the queries of what would spill (float16's two terms, 8-bit
// codes: 6 to 35 registers) are read from LDS in every tile (16 x 8 heads x 8192 positions in groups of 64: float16 of 4 bits 62 ->
// 57 us, of 8 bits, at two blocks before, 88 -> 66, bfloat16 of 8 bits 77 -> 68).
template <typename T, int G> constexpr int attention_blocks() { return sizeof(T) == 4 || G == 4 ? 2 : 3; }
template <typename T, int BITS, int D, int G>
constexpr bool queries_in_lds() {
    constexpr bool f16 = Elem<T>::code != 10;
    return attention_blocks<T, G>() == 3 && D == 128 && (G == 2 ? BITS == 8 || f16 : BITS == 8 && f16);
}

// G groups of a row.  Block: one (batch, key head, split) and 16 / G of its query heads; its wavefronts take tiles of 32 keys in
// turn.
template <typename T, int BITS, int D, int G>
__global__ void __launch_bounds__(64 * kAttnWaves, (attention_blocks<T, G>())) qattn_kernel(const nvq_attention_desc d, const T *__restrict__ q, const uint32_t *__restrict__ kw,
                                                               const T *__restrict__ ks, const T *__restrict__ kb,
                                                               const uint32_t *__restrict__ vw, const T *__restrict__ vs,
                                                               const T *__restrict__ vb, const T *__restrict__ sinks, T *__restrict__ out,
                                                               float *__restrict__ partials) {
    constexpr int TQ = sizeof(T) == 4 ? 3 : Elem<T>::code == 10 ? 1 : 2;  // terms of the queries: exact
    constexpr int TP = 3;                                                 // terms of the weights: 24 bits
    constexpr int R = 16 / G, KS = D / 32, ND = D / 16;  // heads per operand; instructions of K per 16 keys; values of D per lane
    constexpr int kRowBytes = D * BITS / 8, kChunk = kRowBytes / 4, kSlot = BITS * ND;  // bytes of a quarter's codes; bits of a lane's slot
    constexpr bool kWide = sizeof(T) == 4;
    constexpr float kOff = kOffset<BITS, kWide>;
    constexpr float kMiddle = 1 << (BITS - 1);
    constexpr bool kOnes = !kWide;  // (the weights' sum beside the codes)
    constexpr uint32_t kOne = BITS == 8 ? 0x43004300u : BITS == 4 ? 0x41C041C0u : 0x41404140u;  // two of kOff + kMiddle: 128, 24, 12 (at 8, 4, 3 bits)
    constexpr int kHeads = R < 8 ? R : 8;  // (at most eight query heads per key head)
    __shared__ float part[kAttnWaves][kHeads][D + 1];
    __shared__ float wave_m[kAttnWaves][kHeads], wave_l[kAttnWaves][kHeads];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int l = lane & 15, quarter = lane >> 4, g = l / R;
    const int hk = blockIdx.x, b = blockIdx.y;
    const int all = d.query_heads / d.key_heads, S = d.positions;
    // (the blocks of one key head's cache lie gridDim.x * gridDim.y apart: on one XCD where that is a multiple of 8)
    const int parts = (all + R - 1) / R, splits = gridDim.z / parts, first = blockIdx.z % parts * R, split = blockIdx.z / parts;
    const int rep = all - first < R ? all - first : R;  // this block's query heads
    const int64_t row0 = ((int64_t)b * d.key_heads + hk) * S, head0 = (int64_t)b * d.query_heads + hk * all + first;
    const int per = attention_split_keys(S, splits);
    const int s_begin = split * per, s_end = s_begin + per < S ? s_begin + per : S;
    const float scale = d.scale * kLog2e;
    const CodeConstants<BITS> constants;

    // The queries' operands: column (g, head), zeros outside the group; their sums per column.
    const int head = l % R;
    constexpr bool kLdsQueries = queries_in_lds<T, BITS, D, G>();
    __shared__ uint4 queries[kLdsQueries ? KS * TQ : 1][64];  // (the same in all wavefronts)
    uint4 qf[KS][TQ];
    float qsum = 0.0f;
#pragma unroll
    for (int s = 0; s < KS; s++) {
        float v[8];
#pragma unroll
        for (int j = 0; j < 8; j++) {
            const int at = quarter * (D / 4) + 8 * s + code_at<BITS>(j);
            v[j] = head < rep && at / (D / G) == g ? Elem<T>::load(q, (head0 + head) * D + at) : 0.0f;
            qsum += v[j];
        }
        uint32_t t[4][TQ];
#pragma unroll
        for (int j = 0; j < 4; j++) split_pair<TQ>(v[2 * j], v[2 * j + 1], t[j]);
#pragma unroll
        for (int i = 0; i < TQ; i++) {
            qf[s][i] = make_uint4(t[0][i], t[1][i], t[2][i], t[3][i]);
            if (kLdsQueries && wave == 0) queries[s * TQ + i][lane] = qf[s][i];
        }
    }
    if (kLdsQueries) __syncthreads();
    qsum += __shfl_xor(qsum, 16);
    qsum += __shfl_xor(qsum, 32);

    // What a tile of 32 keys reads from memory; the next tile's keys are requested when this one's have become operands, its
    // values likewise.
    constexpr int kRun = G * (int)sizeof(T);  // bytes of a key's scales
    // Float32, four groups: the lane's own group alone (chosen from all of them in registers they went to scratch memory: 16 x 8
    // heads x 8192 positions of 4 bits 459 us, so 76).
    constexpr bool kOwn = kRun == 16;
    struct Quad { uint32_t w[kOwn ? 4 : kRun]; };  // of four consecutive keys
    struct KeyTile {
        uint32_t c[2][(kChunk + 3) / 4];
        Quad s[2], b[2];
    } kt;
    struct ValueTile {
        uint32_t c[8][(kSlot + 31) / 32];
        Quad s[2], b[2];
    } vt;
    const uint8_t *kbytes = reinterpret_cast<const uint8_t *>(kw), *vbytes = reinterpret_cast<const uint8_t *>(vw);
    auto four = [&](const T *p, int key) {
        const uint8_t *at = reinterpret_cast<const uint8_t *>(p + row0 * G);
        Quad o;
        if constexpr (kOwn) {
#pragma unroll
            for (int i = 0; i < 4; i++) o.w[i] = load_any<uint32_t>(at + (int64_t)(key + i < S ? key + i : S - 1) * kRun + 4 * g);
            return o;
        }
        if (key + 4 <= S) {
#pragma unroll
            for (int i = 0; i < kRun; i++) o.w[i] = load_any<uint32_t>(at + (int64_t)key * kRun + 4 * i);
            return o;
        }
#pragma unroll
        for (int i = 0; i < kRun; i++) {  // word i: of key 4 i / kRun, or (one half-precision group) of keys 2 i and 2 i + 1
            if constexpr (kRun >= 4) {
                const int k = key + 4 * i / kRun;
                o.w[i] = load_any<uint32_t>(at + (int64_t)(k < S ? k : S - 1) * kRun + 4 * i % kRun);
            } else {
                const int k0 = key + 2 * i, k1 = k0 + 1;
                o.w[i] = (uint32_t)load_any<uint16_t>(at + (int64_t)(k0 < S ? k0 : S - 1) * 2) |
                         (uint32_t)load_any<uint16_t>(at + (int64_t)(k1 < S ? k1 : S - 1) * 2) << 16;
            }
        }
        return o;
    };
    // A tile that lies inside the cache: the tile's place is a scalar address and the lane's place in it an offset that does not
    // change, so that a load takes no vector instruction for its address; the scales of four keys are one load.  (With an address
    // for every load and key clamped by itself a quarter of the loop's vector instructions were addresses.)
    auto four_inside = [&](const T *p, int s0, int h) __attribute__((always_inline)) {
        const uint8_t *at = reinterpret_cast<const uint8_t *>(p) + (row0 + s0) * kRun;
        Quad o;
        if constexpr (kOwn) {
#pragma unroll
            for (int i = 0; i < 4; i++) o.w[i] = load_any<uint32_t>(at + (uint32_t)(4 * quarter * kRun + 4 * g) + (16 * h + i) * kRun);
        } else {
            o = load_any<Quad>(at + (uint32_t)(4 * quarter * kRun) + 16 * h * kRun);
        }
        return o;
    };
    auto fetch_keys = [&](int s0) __attribute__((always_inline)) {
        if (s0 >= s_end) return;  // (nothing is left for this wavefront)
        if (s0 + kTileKeys <= S) {
            const uint8_t *tile = kbytes + (row0 + s0) * kRowBytes;
#pragma unroll
            for (int h = 0; h < 2; h++) {
                if constexpr (kChunk % 4 == 0) {
                    struct Words { uint32_t w[kChunk / 4]; };
                    const Words w = *reinterpret_cast<const Words *>(tile + (uint32_t)(l * kRowBytes + quarter * kChunk) + 16 * h * kRowBytes);
#pragma unroll
                    for (int i = 0; i < kChunk / 4; i++) kt.c[h][i] = w.w[i];
                } else {  // 6 bytes (16 codes of 3 bits): 8 from where they stay inside the row
                    const int at = quarter * kChunk < kRowBytes - 8 ? quarter * kChunk : kRowBytes - 8;
                    const uint64_t w = load_any<uint64_t>(tile + (uint32_t)(l * kRowBytes + at) + 16 * h * kRowBytes) >> (8 * (quarter * kChunk - at));
                    kt.c[h][0] = (uint32_t)w, kt.c[h][1] = (uint32_t)(w >> 32);
                }
                kt.s[h] = four_inside(ks, s0, h), kt.b[h] = four_inside(kb, s0, h);
            }
            return;
        }
#pragma unroll
        for (int h = 0; h < 2; h++) {
            int key = s0 + 16 * h + l;
            key = key < S ? key : S - 1;  // a key past the end reads the last one and is given no weight
            const uint8_t *row = kbytes + (row0 + key) * kRowBytes;
            if constexpr (kChunk % 4 == 0) {
                struct Words { uint32_t w[kChunk / 4]; };
                const Words w = *reinterpret_cast<const Words *>(row + quarter * kChunk);
#pragma unroll
                for (int i = 0; i < kChunk / 4; i++) kt.c[h][i] = w.w[i];
            } else {  // 6 bytes (16 codes of 3 bits): 8 from where they stay inside the row
                const int at = quarter * kChunk < kRowBytes - 8 ? quarter * kChunk : kRowBytes - 8;
                const uint64_t w = load_any<uint64_t>(row + at) >> (8 * (quarter * kChunk - at));
                kt.c[h][0] = (uint32_t)w, kt.c[h][1] = (uint32_t)(w >> 32);
            }
            kt.s[h] = four(ks, s0 + 16 * h + 4 * quarter), kt.b[h] = four(kb, s0 + 16 * h + 4 * quarter);
        }
    };
    // the lane's slot of a row at `row` + `lanes`, `lanes` without the slot's own place
    auto value_slot = [&](const uint8_t *row, uint32_t lanes, int j) __attribute__((always_inline)) {
        if constexpr (kSlot == 64) {
            const uint2 w = *reinterpret_cast<const uint2 *>(row + (lanes + 8 * l));
            vt.c[j][0] = w.x, vt.c[j][1] = w.y;
        } else if constexpr (kSlot == 32) {
            vt.c[j][0] = *reinterpret_cast<const uint32_t *>(row + (lanes + 4 * l));
        } else if constexpr (kSlot == 16) {
            vt.c[j][0] = *reinterpret_cast<const uint16_t *>(row + (lanes + 2 * l));
        } else if constexpr (kSlot == 24) {
            vt.c[j][0] = load_any<uint32_t>(row + (lanes + 3 * l - (l == 15))) >> (l == 15 ? 8 : 0);
        } else {  // 12 bits
            vt.c[j][0] = load_any<uint16_t>(row + (lanes + 3 * l / 2)) >> (4 * (l & 1));
        }
    };
    auto fetch_values = [&](int s0) __attribute__((always_inline)) {
        if (s0 >= s_end) return;
        if (s0 + kTileKeys <= S) {
            const uint8_t *tile = vbytes + (row0 + s0) * kRowBytes;
#pragma unroll
            for (int j = 0; j < 8; j++) value_slot(tile + (16 * (j >> 2) + (j & 3)) * kRowBytes, 4 * quarter * kRowBytes, j);
#pragma unroll
            for (int h = 0; h < 2; h++) vt.s[h] = four_inside(vs, s0, h), vt.b[h] = four_inside(vb, s0, h);
            return;
        }
#pragma unroll
        for (int j = 0; j < 8; j++) {
            const int key = s0 + 16 * (j >> 2) + 4 * quarter + (j & 3);
            value_slot(vbytes + (row0 + (key < S ? key : S - 1)) * kRowBytes, 0, j);
        }
#pragma unroll
        for (int h = 0; h < 2; h++) vt.s[h] = four(vs, s0 + 16 * h + 4 * quarter), vt.b[h] = four(vb, s0 + 16 * h + 4 * quarter);
    };
    // The lane's own group of key i.
    const int down = 16 * (g & 1);
    const uint32_t half = g & 1 ? 0x03020C0Cu : 0x01000C0Cu;  // (its 16 bits above zeros: one byte permutation)
    auto pick = [&](const Quad &o, int i) {
        if constexpr (kOwn) {
            return u2f(o.w[i]);
        } else if constexpr (sizeof(T) == 4) {
            uint32_t w = o.w[G * i];
#pragma unroll
            for (int e = 1; e < G; e++) w = g == e ? o.w[G * i + e] : w;
            return u2f(w);
        } else {
            uint32_t w = o.w[G * i / 2];
            if constexpr (G == 4) w = g >= 2 ? o.w[2 * i + 1] : w;
            if constexpr (Elem<T>::code == 10) {
                if constexpr (G == 1) return u2f(i & 1 ? w & 0xFFFF0000u : w << 16);
                return u2f(__builtin_amdgcn_perm(0u, w, half));
            } else {
                return (float)__builtin_bit_cast(f16_t, (uint16_t)(w >> (G == 1 ? 16 * (i & 1) : down)));
            }
        }
    };

    floatx4_t acc[ND], ones = {0.0f, 0.0f, 0.0f, 0.0f};
    float m = -1.0e30f, denom = 0.0f, accb = 0.0f;
#pragma unroll
    for (int i = 0; i < ND; i++) acc[i] = floatx4_t{0.0f, 0.0f, 0.0f, 0.0f};
    fetch_keys(s_begin + wave * kTileKeys);
    fetch_values(s_begin + wave * kTileKeys);
    for (int s0 = s_begin + wave * kTileKeys; s0 < s_end; s0 += kAttnWaves * kTileKeys) {
        float score[8];
        if constexpr (kLdsQueries) {
            asm volatile("" ::: "memory");  // (not kept from the tile before)
#pragma unroll
            for (int s = 0; s < KS; s++)
#pragma unroll
                for (int i = 0; i < TQ; i++) qf[s][i] = queries[s * TQ + i][lane];
        }
#pragma unroll
        for (int h = 0; h < 2; h++) {
            floatx4_t sum = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
            for (int s = 0; s < KS; s++) {
                uint4 kf;
                if constexpr (BITS == 8) {
                    kf = eight_codes<8, kWide>(constants, kt.c[h][2 * s], kt.c[h][2 * s + 1]);
                } else if constexpr (BITS == 4) {
                    kf = eight_codes<4, kWide>(constants, kt.c[h][s], 0);
                } else {
                    constexpr int W = (kChunk + 3) / 4;
                    const int bit = 24 * s, w = bit / 32, sh = bit % 32;
                    kf = eight_codes<3, kWide>(constants, sh == 0 ? kt.c[h][w] : __builtin_amdgcn_alignbit(kt.c[h][w + 1 < W ? w + 1 : w], kt.c[h][w], sh), 0);
                }
#pragma unroll
                for (int i = 0; i < TQ; i++) sum = mfma16(kf, qf[s][i], sum);
            }
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const float sk = pick(kt.s[h], r), bk = pick(kt.b[h], r);
                float v = __builtin_fmaf(sk, sum[r], __builtin_fmaf(-kOff, sk, bk) * qsum);
                // the groups of a row: columns R apart
                if constexpr (G == 4) v += u2f((uint32_t)__builtin_amdgcn_mov_dpp((int)f2u(v), 0x124, 0xF, 0xF, true));
                if constexpr (G >= 2) v += u2f((uint32_t)__builtin_amdgcn_mov_dpp((int)f2u(v), 0x128, 0xF, 0xF, true));
                score[4 * h + r] = v * scale;
            }
        }
        if (s0 + kTileKeys > s_end) {
            asm volatile("");  // (a branch: as selects it would cost every tile)
#pragma unroll
            for (int j = 0; j < 8; j++)
                if (s0 + 16 * (j >> 2) + 4 * quarter + (j & 3) >= s_end) score[j] = -INFINITY;
        }
        fetch_keys(s0 + kAttnWaves * kTileKeys);
        float top = score[0];
#pragma unroll
        for (int j = 1; j < 8; j++) top = fmaxf(top, score[j]);
        // The sums are rescaled only when a maximum has grown by more than 2^8; until then weights are at most 2^8.
        if (__any(top > m + 8.0f)) {
            top = fmaxf(top, __shfl_xor(top, 16));
            top = fmaxf(top, __shfl_xor(top, 32));
            const float m_new = fmaxf(m, top), f = exp2f(m - m_new);
            m = m_new, denom *= f, accb *= f;
#pragma unroll
            for (int r = 0; r < 4; r++) {
                ones[r] *= f;
#pragma unroll
                for (int i = 0; i < ND; i++) acc[i][r] *= f;
            }
        }
        float w[8];
#pragma unroll
        for (int j = 0; j < 8; j++) {
            const float p = __builtin_amdgcn_exp2f(score[j] - m);
            denom += p;
            const float sv = pick(vt.s[j >> 2], j & 3), bv = pick(vt.b[j >> 2], j & 3);
            accb = __builtin_fmaf(p, __builtin_fmaf(kMiddle, sv, bv), accb);
            w[j] = p * sv;
        }
        uint32_t t[4][TP];
        uint4 pf[TP];
#pragma unroll
        for (int j = 0; j < 4; j++) split_pair<TP>(w[2 * j], w[2 * j + 1], t[j]);
#pragma unroll
        for (int e = 0; e < TP; e++) {
            pf[e] = make_uint4(t[0][e], t[1][e], t[2][e], t[3][e]);
            if constexpr (kOnes) ones = mfma16(make_uint4(kOne, kOne, kOne, kOne), pf[e], ones);
        }
        // value i of the lane's slot, two keys a word
#pragma unroll
        for (int i = 0; i < ND; i++) {
            uint32_t p[4];
#pragma unroll
            for (int j = 0; j < 4; j++) {
                if constexpr (kWide) {
                    const int w = BITS * i / 32, sh = BITS * i % 32;  // (a code of 3 bits: within the slot's 12 or 24)
                    constexpr uint32_t mask = (1u << BITS) - 1u;
                    p[j] = pack_exact((float)((vt.c[2 * j][w] >> sh) & mask) + kOff, (float)((vt.c[2 * j + 1][w] >> sh) & mask) + kOff);
                } else if constexpr (BITS == 8) {
                    const int w = i / 4;
                    const uint32_t x = vt.c[2 * j][w] >> (8 * (i % 4)), y = vt.c[2 * j + 1][w] >> (8 * (i % 4));
                    p[j] = pack_exact((float)(x & 0xFFu), (float)(y & 0xFFu));
                } else {
                    // sixteen bits of each key that hold the code, side by side
                    const bool high = BITS * i + BITS > 16;
                    const int from = BITS == 4 ? 16 : 8;  // the second piece's first bit
                    const uint32_t sel = !high ? 0x05040100u : BITS == 4 ? 0x07060302u : 0x06050201u;
                    const uint32_t both = __builtin_amdgcn_perm(vt.c[2 * j + 1][0], vt.c[2 * j][0], sel);
                    p[j] = two_codes(constants, both, BITS * i - (high ? from : 0));
                }
            }
            const uint4 vf = make_uint4(p[0], p[1], p[2], p[3]);
#pragma unroll
            for (int e = 0; e < TP; e++) acc[i] = mfma16(vf, pf[e], acc[i]);
        }
        fetch_values(s0 + kAttnWaves * kTileKeys);
    }

    // merge: the block's maximum, every wavefront scaled to it, the wavefronts added up
    denom += __shfl_xor(denom, 16), accb += __shfl_xor(accb, 16);
    denom += __shfl_xor(denom, 32), accb += __shfl_xor(accb, 32);
    if (head < rep) {
        if (lane < R) wave_m[wave][head] = m, wave_l[wave][head] = denom;
#pragma unroll
        for (int i = 0; i < ND; i++)
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const int at = ND * (4 * quarter + r) + i;  // of D: this column's group has it or another column's
                // (the operands and kOff + kMiddle alone went through the same sums)
                if (at / (D / G) == g) part[wave][head][at] = acc[i][r] - (kOnes ? ones[r] : 0.0f) + accb;
            }
    }
    __syncthreads();
    for (int e = tid; e < rep * D; e += 64 * kAttnWaves) {
        const int hd = e / D, at = e % D;
        float top = -1.0e30f;
#pragma unroll
        for (int w = 0; w < kAttnWaves; w++) top = fmaxf(top, wave_m[w][hd]);
        float sum = 0.0f, total = 0.0f;
#pragma unroll
        for (int w = 0; w < kAttnWaves; w++) {
            const float f = exp2f(wave_m[w][hd] - top);
            total = __builtin_fmaf(wave_l[w][hd], f, total);
            sum = __builtin_fmaf(part[w][hd][at], f, sum);
        }
        if (splits == 1) {
            if (sinks != nullptr) {
                const float sink = Elem<T>::load(sinks, hk * all + first + hd) * kLog2e, t2 = fmaxf(top, sink), f = exp2f(top - t2);
                sum *= f, total = total * f + exp2f(sink - t2);
            }
            Elem<T>::store(out, (head0 + hd) * D + at, sum / total);
        } else {  // this split's state: maximum (of base-2 scores), denominator, weighted sum
            float *dst = partials + ((head0 + hd) * splits + split) * (D + 2);
            if (at == 0) dst[0] = top, dst[1] = total;
            dst[2 + at] = sum;
        }
    }
}

// ── one query head of a key head at a time, on the vector units ─────────────────────────────────────────────────────
// A row of the cache is CH chunks of 32 codes (16 of 8 bits: 16 bytes); lane l of a wavefront takes chunk l % CH of key l / CH of
// the wavefront's tile of 64 / CH keys, so that its loads read consecutive rows.  The lanes of a key add their partial dot products,
// every lane keeps the softmax of the keys it has seen and its chunk of the output, and the states of a block meet in LDS.
template <int BITS> struct Chunk { uint32_t w[BITS == 3 ? 3 : 4]; };

template <int BITS>
__device__ __forceinline__ Chunk<BITS> load_chunk(const uint32_t *p) {
    Chunk<BITS> c;
    if constexpr (BITS == 3) {
        c.w[0] = p[0], c.w[1] = p[1], c.w[2] = p[2];  // (rows of 3-bit codes are whole dwords: 4-byte aligned)
    } else {
        const uint4 v = *reinterpret_cast<const uint4 *>(p);
        c.w[0] = v.x, c.w[1] = v.y, c.w[2] = v.z, c.w[3] = v.w;
    }
    return c;
}

// Code i of a chunk as a float (i is a constant after unrolling).
template <int BITS>
__device__ __forceinline__ float chunk_code(const Chunk<BITS> &c, int i) {
    if constexpr (BITS == 4) {
        return (float)((c.w[i >> 3] >> (4 * (i & 7))) & 15u);
    } else if constexpr (BITS == 8) {
        return (float)((c.w[i >> 2] >> (8 * (i & 3))) & 255u);
    } else {
        const int bit = 3 * i, dw = bit >> 5, sh = bit & 31;
        const uint32_t v = sh <= 29 ? c.w[dw] >> sh : (c.w[dw] >> sh) | (c.w[dw + 1] << (32 - sh));
        return (float)(v & 7u);
    }
}

template <typename T, int BITS, int D>
__global__ void __launch_bounds__(64 * kAttnWaves) qattn_vector_kernel(const nvq_attention_desc d, const T *__restrict__ q, const uint32_t *__restrict__ kw,
                                                                      const T *__restrict__ ks, const T *__restrict__ kb,
                                                                      const uint32_t *__restrict__ vw, const T *__restrict__ vs,
                                                                      const T *__restrict__ vb, const T *__restrict__ sinks, T *__restrict__ out,
                                                                      float *__restrict__ partials) {
    constexpr int CPL = BITS == 8 ? 16 : 32;  // codes of a lane
    constexpr int CW = CPL * BITS / 32;       // their dwords
    constexpr int CH = D / CPL;               // lanes of a key: 2, 4 or 8
    constexpr int KPT = 64 / CH;              // keys of a wavefront's tile
    constexpr int kSlots = KPT * kAttnWaves;
    // float32: sums over codes from the middle of their range, as above; the output's rounding covers the 16-bit types' sums
    constexpr float kMiddle = sizeof(T) == 4 ? (float)(1 << (BITS - 1)) : 0.0f;
    __shared__ float part[kSlots][D + 1];
    __shared__ float slot_m[kSlots], slot_l[kSlots];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int c = lane % CH, j = lane / CH;
    const int h = blockIdx.x, b = blockIdx.y;
    const int rep = d.query_heads / d.key_heads, hk = h / rep;
    const int S = d.positions, groups = D / d.group_size;
    const int gi = (c * CPL) / d.group_size;  // (a chunk lies inside one group)
    const int64_t row0 = ((int64_t)b * d.key_heads + hk) * S, head = (int64_t)b * d.query_heads + h;
    const int splits = gridDim.z, per = attention_split_keys(S, splits);
    const int s_begin = blockIdx.z * per, s_end = s_begin + per < S ? s_begin + per : S;
    const float scale = d.scale * kLog2e;

    float qv[CPL], qs[4] = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int i = 0; i < CPL; i++) qv[i] = Elem<T>::load(q, head * D + c * CPL + i), qs[i & 3] += qv[i];
    const float qsum = (qs[0] + qs[1]) + (qs[2] + qs[3]);
    float m = -1.0e30f, l = 0.0f, acc[CPL], accb = 0.0f;
#pragma unroll
    for (int i = 0; i < CPL; i++) acc[i] = 0.0f;

    struct Tile {
        Chunk<BITS> kc, vc;
        T sk, bk, sv, bv;
    };
    auto fetch = [&](int s0) {
        const int s = s0 + j;
        const int64_t r = row0 + (s < s_end ? s : S - 1);  // a key past the end reads the last one and is given no weight
        Tile t;
        t.kc = load_chunk<BITS>(kw + (r * CH + c) * CW), t.vc = load_chunk<BITS>(vw + (r * CH + c) * CW);
        t.sk = ks[r * groups + gi], t.bk = kb[r * groups + gi], t.sv = vs[r * groups + gi], t.bv = vb[r * groups + gi];
        return t;
    };
    Tile cur = fetch(s_begin + wave * KPT);
    for (int s0 = s_begin + wave * KPT; s0 < s_end; s0 += kAttnWaves * KPT) {
        const Tile nxt = fetch(s0 + kAttnWaves * KPT);  // requested before this one is computed
        const float sk = Elem<T>::load(&cur.sk, 0), bk = __builtin_fmaf(kMiddle, sk, Elem<T>::load(&cur.bk, 0));
        const float sv = Elem<T>::load(&cur.sv, 0), bv = __builtin_fmaf(kMiddle, sv, Elem<T>::load(&cur.bv, 0));
        float dot[4] = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int i = 0; i < CPL; i++) dot[i & 3] = __builtin_fmaf(qv[i], chunk_code<BITS>(cur.kc, i) - kMiddle, dot[i & 3]);
        float score = __builtin_fmaf(sk, (dot[0] + dot[1]) + (dot[2] + dot[3]), bk * qsum);
#pragma unroll
        for (int o = 1; o < CH; o <<= 1) score += __shfl_xor(score, o);  // the lanes of a key sit side by side
        score = s0 + j < s_end ? score * scale : -INFINITY;
        if (__any(score > m + 8.0f)) {
            const float m_new = fmaxf(m, score), f = exp2f(m - m_new);
            m = m_new, l *= f, accb *= f;
#pragma unroll
            for (int i = 0; i < CPL; i++) acc[i] *= f;
        }
        const float p = __builtin_amdgcn_exp2f(score - m), pv = p * sv;
        l += p;
        accb = __builtin_fmaf(p, bv, accb);
#pragma unroll
        for (int i = 0; i < CPL; i++) acc[i] = __builtin_fmaf(pv, chunk_code<BITS>(cur.vc, i) - kMiddle, acc[i]);
        cur = nxt;
    }

    // merge: the block's maximum, every slot scaled to it, the slots added up by 256 / D groups of threads in four chains each
    constexpr int kGroups = 64 * kAttnWaves / D;
    __shared__ float sums[kGroups][D], denoms[kGroups];
    const int slot = wave * KPT + j;
    if (c == 0) slot_m[slot] = m;
    __syncthreads();
    float top = lane < kSlots ? slot_m[lane] : -1.0e30f;
    if constexpr (kSlots == 128) top = fmaxf(top, slot_m[lane + 64]);
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) top = fmaxf(top, __shfl_xor(top, o));
    const float w = exp2f(m - top);
    if (c == 0) slot_l[slot] = l * w;
#pragma unroll
    for (int i = 0; i < CPL; i++) part[slot][c * CPL + i] = (acc[i] + accb) * w;
    __syncthreads();
    const int at = tid % D, group = tid / D;
    float dn[4] = {0.0f, 0.0f, 0.0f, 0.0f}, sm[4] = {0.0f, 0.0f, 0.0f, 0.0f};
    for (int t = group * (kSlots / kGroups); t < (group + 1) * (kSlots / kGroups); t += 4)
#pragma unroll
        for (int u = 0; u < 4; u++) dn[u] += slot_l[t + u], sm[u] += part[t + u][at];
    sums[group][at] = (sm[0] + sm[1]) + (sm[2] + sm[3]);
    if (at == 0) denoms[group] = (dn[0] + dn[1]) + (dn[2] + dn[3]);
    __syncthreads();
    if (group != 0) return;
    float sum = sums[0][at] + sums[1][at], denom = denoms[0] + denoms[1];
    if constexpr (kGroups == 4) sum += sums[2][at] + sums[3][at], denom += denoms[2] + denoms[3];
    if (splits == 1) {
        if (sinks != nullptr) {
            const float sink = Elem<T>::load(sinks, h) * kLog2e, t2 = fmaxf(top, sink), f = exp2f(top - t2);
            sum *= f, denom = denom * f + exp2f(sink - t2);
        }
        Elem<T>::store(out, head * D + at, sum / denom);
    } else {
        float *dst = partials + (head * splits + blockIdx.z) * (D + 2);
        if (at == 0) dst[0] = top, dst[1] = denom;
        dst[2 + at] = sum;
    }
}

// The splits of one (batch, head) merged.
template <typename T, int D>
__global__ void __launch_bounds__(kMergeParts * D) qattn_merge_kernel(const nvq_attention_desc d, const float *__restrict__ partials, int splits,
                                                                      const T *__restrict__ sinks, T *__restrict__ out) {
    const int64_t head = (int64_t)blockIdx.y * d.query_heads + blockIdx.x;
    merge_attention_states<T, D>(partials + head * splits * (D + 2), D + 2, splits, sinks != nullptr,
                                 sinks != nullptr ? Elem<T>::load(sinks, blockIdx.x) * kLog2e : 0.0f, out + head * D);
}

// The same for few splits, D / 4 threads a head.
template <typename T, int D>
__global__ void __launch_bounds__(64) qattn_merge_few_kernel(const nvq_attention_desc d, const float *__restrict__ partials, int splits,
                                                             const T *__restrict__ sinks, T *__restrict__ out) {
    const int64_t h = (int64_t)blockIdx.x * (256 / D) + (int)threadIdx.x / (D / 4), head = (int64_t)blockIdx.y * d.query_heads + h;
    if (h >= d.query_heads) return;
    merge_few_states<T, D>(partials + head * splits * (D + 2), D + 2, splits, sinks != nullptr, sinks != nullptr ? Elem<T>::load(sinks, h) * kLog2e : 0.0f,
                           out + head * D, (int)threadIdx.x % (D / 4) * 4);
}

struct Plan {
    bool vector;
    int splits;  // of the positions over the grid
};
Plan attention_plan(const nvq_attention_desc &d);

struct Operands {
    const void *q, *kw, *ks, *kb, *vw, *vs, *vb, *sinks;
    void *out, *workspace;
};

template <typename T, typename K>
void start_attention(K kernel, dim3 grid, const nvq_attention_desc &d, const Operands &o, hipStream_t s) {
    hipLaunchKernelGGL(kernel, grid, dim3(64 * kAttnWaves), 0, s, d, (const T *)o.q, (const uint32_t *)o.kw, (const T *)o.ks, (const T *)o.kb,
                       (const uint32_t *)o.vw, (const T *)o.vs, (const T *)o.vb, (const T *)o.sinks, (T *)o.out, (float *)o.workspace);
}

template <typename T, int BITS, int D>
int32_t run_attention_sized(const nvq_attention_desc &d, const Operands &o, hipStream_t s) {
    Plan p = attention_plan(d);
    if (o.workspace == nullptr) p.splits = 1;
    if (p.vector) {
        start_attention<T>(qattn_vector_kernel<T, BITS, D>, dim3((unsigned)d.query_heads, (unsigned)d.batch, (unsigned)p.splits), d, o, s);
    } else {
        const int groups = D / d.group_size, heads = 16 / groups;  // (groups have 32 values at least)
        const int64_t parts = (d.query_heads / d.key_heads + heads - 1) / heads;
        const dim3 grid((unsigned)d.key_heads, (unsigned)d.batch, (unsigned)(p.splits * parts));
        if (groups == 1) start_attention<T>(qattn_kernel<T, BITS, D, 1>, grid, d, o, s);
        else if (groups == 2) start_attention<T>(qattn_kernel<T, BITS, D, 2>, grid, d, o, s);
        else if constexpr (D == 128) start_attention<T>(qattn_kernel<T, BITS, D, 4>, grid, d, o, s);
    }
    NVQ_LAUNCH_CHECK("quantized_attention");
    if (p.splits > 1) {
        if (p.splits <= kFewSplits)
            hipLaunchKernelGGL((qattn_merge_few_kernel<T, D>), dim3((unsigned)((d.query_heads + 256 / D - 1) / (256 / D)), (unsigned)d.batch), dim3(64), 0, s, d,
                               (const float *)o.workspace, p.splits, (const T *)o.sinks, (T *)o.out);
        else
            hipLaunchKernelGGL((qattn_merge_kernel<T, D>), dim3((unsigned)d.query_heads, (unsigned)d.batch), dim3(kMergeParts * D), 0, s, d,
                           (const float *)o.workspace, p.splits, (const T *)o.sinks, (T *)o.out);
        NVQ_LAUNCH_CHECK("quantized_attention merge");
    }
    return NVQ_OK;
}

template <typename T, int BITS>
int32_t run_attention(const nvq_attention_desc &d, const Operands &o, hipStream_t s) {
    return d.head_dim == 64 ? run_attention_sized<T, BITS, 64>(d, o, s) : run_attention_sized<T, BITS, 128>(d, o, s);
}

template <typename T>
int32_t run_attention_bits(const nvq_attention_desc &d, const Operands &o, hipStream_t s) {
    return d.bits == 4 ? run_attention<T, 4>(d, o, s) : d.bits == 3 ? run_attention<T, 3>(d, o, s) : run_attention<T, 8>(d, o, s);
}

// Both kernels as timed on 592 calls (1 to 8 query heads per key head, 128 to 20000 positions, batches of 1 to 32, 3, 4 and 8 bits in
// groups of 32 and 64, head sizes 64 and 128, the three types): the vector kernel's time grows with the query heads, the other's
// with the key heads (times the blocks that share one), and the vector kernel starts sooner.  Per thousand positions of a head
// of 128 values it takes 0.0245 us a query head (0.033 with 8 bits), the matrix cores 0.060 (0.047 in float32).  Choosing by them
// is 0.4 % above always taking the faster kernel, 1.28 x at worst.  us, vector / matrix cores, 16 x 8 key heads x 8192 positions,
// bfloat16, 4-bit groups of 64: one query head 40 / 60, two 71 / 58, four 116 / 56; 32 x 4 x 300: 7.4 / 10.6, 8 / 10.8, 10 / 11.1.
bool vector_is_faster(const nvq_attention_desc &d) {
    const double rep = (double)d.query_heads / (double)d.key_heads, parts = ceil(rep * (double)d.head_dim / (16.0 * d.group_size));
    const double positions = (double)d.batch * (double)d.key_heads * (double)d.positions * (double)d.head_dim / 128.0e3;
    return (d.bits == 8 ? 0.033 : 0.0245) * rep * positions < (d.bits == 8 ? 3.0 : 1.5) + (d.dtype == NVQ_F32 ? 0.047 : 0.060) * parts * positions;
}

// Splits of the positions over the grid, at most 64 (a lane each when they are merged).  Matrix cores: three blocks of four
// wavefronts per compute unit, at least two tiles a wavefront; vector: two blocks, at least 256 keys.
Plan attention_plan(const nvq_attention_desc &d) {
    Plan p{vector_is_faster(d), 1};
    const int64_t heads = d.batch * (p.vector ? d.query_heads : d.key_heads), units = compute_units();
    if (heads <= 0 || (p.vector && d.positions < 512)) return p;
    int64_t want = p.vector ? (2 * units + heads - 1) / heads : 3 * units / heads;
    const int64_t most = d.positions / (2 * kAttnWaves * kTileKeys);
    want = want > most ? most : want;
    want = want > 64 ? 64 : want;
    if (want < 2) return p;
    const int per = attention_split_keys(d.positions, (int)want);  // whole tiles: fewer splits may cover the positions
    p.splits = (int)((d.positions + per - 1) / per);
    return p;
}

}  // namespace

size_t attention_workspace_bytes(const nvq_attention_desc &d) {
    const int splits = attention_plan(d).splits;
    return splits > 1 ? (size_t)d.batch * (size_t)d.query_heads * (size_t)splits * (size_t)(d.head_dim + 2) * sizeof(float) : 0;
}

int32_t launch_quantized_attention(const nvq_attention_desc &d, const void *q, const void *kw, const void *ks, const void *kb,
                                   const void *vw, const void *vs, const void *vb, const void *sinks, void *out, void *workspace,
                                   hipStream_t s) {
    const Operands o{q, kw, ks, kb, vw, vs, vb, sinks, out, workspace};
    switch (d.dtype) {
    case NVQ_F32: return run_attention_bits<float>(d, o, s);
    case NVQ_BF16: return run_attention_bits<bf16_t>(d, o, s);
    default: return run_attention_bits<f16_t>(d, o, s);
    }
}

}  // namespace nvq
