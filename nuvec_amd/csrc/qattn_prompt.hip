// Attention of several query rows per head over an affine-quantized key / value cache on the gfx950 matrix cores: the
// prompt's side of the reference's `quantized_attention` (crates/nuvec-core/src/fast/imp.rs:3996-4035, the composition of two
// quantized products and a softmax; nuvec-lm's causal mask, crates/nuvec-lm/src/model.rs:3646-3700):
//     out[b, h, i, :] = softmax(scale * q[b, h, i, :] . K[b, h / rep]^T [masked] [, sink[h]]) . V[b, h / rep]
// with the scores and the softmax in float32 and never in memory; values and the softmax's weights are rounded to the
// element type once before their products, and keys where the composition's product rounds them (twice there: the CPU's weights).
// Where that holds them in float32 they are two terms of the element type (keys_are_two_terms): exact wherever scale and bias lie as
// close as `quantize` leaves them, 17 or 23 bits at least.
//
// Two kernels.  The first dequantizes the cache once into a workspace (a cache of 2048 positions x 8 heads is 8 MB there, and
// stays in the chip's caches; every tile of query rows reads all of it), laid out as the operands of the matrix instruction:
// a wavefront's load is 1 KB of consecutive bytes and no kernel transposes anything.  The second walks it with an online
// softmax.
//
// The rows of a key head are its rep x L query rows (row r: query r / rep, head r % rep), so that grouped heads and a few
// queries share tiles.  A wavefront owns 32 rows and forms the scores transposed, S^T = K . Q^T with v_mfma_32x32x16: a lane
// then holds 16 of 32 keys of ONE row, its maximum and sum are in-lane but for one exchange, and the weights are already the
// operand of O^T = V^T . P^T - the contraction's order is free, so V's keys are stored in the order the lanes hold them (lane
// half h has keys 4 h + {0..3} and 8 + 4 h + {0..3} of sixteen).
//
// What fills the chip: few rows are walked by several wavefronts of a block, each taking every KP-th tile of keys, and where
// even that leaves compute units idle by several blocks whose float32 states a third kernel merges.
#include "attention_merge.h"
#include "nvq_device.h"
#include "nvq_internal.h"
#include "qmf_kernel.h"

namespace nvq {
namespace {

using qmf::floatx16_t;
using qmf::Ops;

constexpr int kKeys = 32;       // keys of a tile
constexpr int kRows = 32;       // rows of a wavefront
constexpr int kWaves = 4;       // wavefronts of a block: row groups x parts of the keys
constexpr float kLog2e = 1.44269504088896340736f;

struct PromptArgs {
    const void *q;
    const uint4 *keys, *values;  // operands of the heads from head0 on, [heads][tiles][terms of the keys][D / 16 x 64]
    const void *sinks;
    void *out;
    float *partials;             // [splits][heads x queries][D + 2] or NULL
    float scale;
    int32_t causal;
    int32_t query_heads, key_heads, rep, queries, positions;
    int32_t head0;               // (batch x key head) of the launch's first
    int32_t tiles, row_tiles, splits;
};

// Eight codes, each value rounded once: the product's own rounding first, as `dequantize` has it, is the larger of the two (error
// against float64, 64 queries over 1024 positions of 8 bits: float16 8.7e-4 with both, 4.0e-4 with one, 8.3e-4 in the composition;
// bfloat16 7.2e-3, 3.2e-3, 8.3e-3).  TERMS 2: what that leaves in a second term (the first is finite, so that an infinity is the
// second's).
template <typename T, int BITS, int TERMS>
__device__ __forceinline__ void dequantize_eight(uint64_t codes, float s, float b, uint4 (&out)[TERMS]) {
    constexpr float most = Elem<T>::code == NVQ_BF16 ? 3.38953139e38f : 65504.0f;
    auto at = [&](int i) { return __builtin_fmaf((float)(uint32_t)((codes >> (i * BITS)) & ((1u << BITS) - 1u)), s, b); };
    uint32_t p[TERMS][4];
#pragma unroll
    for (int i = 0; i < 4; i++) {
        float v0 = at(2 * i), v1 = at(2 * i + 1);
        if constexpr (TERMS == 2) {
            p[0][i] = Ops<T>::pack(__builtin_amdgcn_fmed3f(v0, -most, most), __builtin_amdgcn_fmed3f(v1, -most, most));
            v0 -= qmf::half_lo<T>(p[0][i]), v1 -= qmf::half_hi<T>(p[0][i]);
        }
        p[TERMS - 1][i] = Ops<T>::pack(v0, v1);
    }
#pragma unroll
    for (int t = 0; t < TERMS; t++) out[t] = make_uint4(p[t][0], p[t][1], p[t][2], p[t][3]);
}

// Block: one tile of 32 keys of one (batch, key head); positions past the end are zeros.  Bound by the latency of its requests: codes,
// scales and biases of 32 rows are runs of consecutive bytes and pass through LDS (eight codes a lane straight from 32 rows, and its
// scale: sixteen requests a wavefront of 32 cache lines each, 7.6 us for 2048 positions x 8 heads of 8 bits instead of 6.2).
template <typename T, int BITS, int D, int TERMS>
__global__ void __launch_bounds__(256) prompt_operands_kernel(const uint32_t *__restrict__ kw, const T *__restrict__ ks, const T *__restrict__ kb,
                                                             const uint32_t *__restrict__ vw, const T *__restrict__ vs, const T *__restrict__ vb,
                                                             int head0, int positions, int group_shift, uint4 *__restrict__ keys, uint4 *__restrict__ values) {
    constexpr int kChunks = kKeys * D / 8, words = D * BITS / 32, kWords = kKeys * words, kOwn = (kWords + 255) / 256;
    constexpr int kStride = words + 1 + words % 2;  // dwords of a row in LDS, an odd number: lanes of one column fall on different banks
    __shared__ __align__(16) uint16_t tile[kKeys][D + 8];
    __shared__ uint32_t codes[2][kKeys * kStride + 1];
    __shared__ T scales[4][kKeys * (D / 32)];
    const int tid = threadIdx.x;
    const int64_t block = (int64_t)blockIdx.y * gridDim.x + blockIdx.x;
    const int groups = D >> group_shift, s0 = blockIdx.x * kKeys, rows = positions - s0 < kKeys ? positions - s0 : kKeys;
    const int64_t row0 = (int64_t)(head0 + blockIdx.y) * positions + s0;
    const uint32_t *kcodes = kw + row0 * words, *vcodes = vw + row0 * words;
    uint32_t kc[kOwn], vc[kOwn];
#pragma unroll
    for (int u = 0; u < kOwn; u++) {  // (past the end: the last dword, not used)
        const int i = 256 * u + tid < rows * words ? 256 * u + tid : rows * words - 1;
        kc[u] = kcodes[i], vc[u] = vcodes[i];
    }
    // scales, biases of the keys, then of the values: 64 threads each
    const int kind = tid >> 6, first = tid & 63;
    const T *from = (kind == 0 ? ks : kind == 1 ? kb : kind == 2 ? vs : vb) + row0 * groups;
    T sc[kKeys * (D / 32) / 64];
#pragma unroll
    for (int u = 0; u < kKeys * (D / 32) / 64; u++) {
        const int i = first + 64 * u;
        sc[u] = from[i < rows * groups ? i : rows * groups - 1];
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int u = 0; u < kOwn; u++) {
        const int i = 256 * u + tid;
        if ((u + 1) * 256 <= kWords || i < kWords) codes[0][i / words * kStride + i % words] = kc[u], codes[1][i / words * kStride + i % words] = vc[u];
    }
#pragma unroll
    for (int u = 0; u < kKeys * (D / 32) / 64; u++) scales[kind][first + 64 * u] = sc[u];
    __syncthreads();
#pragma unroll
    for (int c0 = 0; c0 < kChunks; c0 += 256) {
        const int c = c0 + tid, key = c & 31, d0 = (c >> 5) * 8;  // (chunk (step << 6 | half << 5 | key): values 16 step + 8 half ..)
        const int byte = d0 / 8 * BITS, w = key * kStride + (byte >> 2), g = key * groups + (d0 >> group_shift);
        auto eight = [&](const uint32_t *of) {  // (BITS bytes from byte 0 .. 3 of a word: they end in the second one)
            uint64_t v = of[w];
            if constexpr (BITS > 1 && BITS != 4) v |= (uint64_t)of[w + 1] << 32;
            return v >> (8 * (byte & 3));
        };
        uint4 k[TERMS] = {}, v[1] = {};
        if (key < rows) {
            dequantize_eight<T, BITS, TERMS>(eight(codes[0]), Elem<T>::load(scales[0], g), Elem<T>::load(scales[1], g), k);
            dequantize_eight<T, BITS, 1>(eight(codes[1]), Elem<T>::load(scales[2], g), Elem<T>::load(scales[3], g), v);
        }
#pragma unroll
        for (int t = 0; t < TERMS; t++) keys[(block * TERMS + t) * kChunks + c] = k[t];
        *reinterpret_cast<uint4 *>(&tile[key][d0]) = v[0];
    }
    __syncthreads();
#pragma unroll
    for (int c0 = 0; c0 < kChunks; c0 += 256) {
        const int c = c0 + tid, lane = c & 63, h = lane >> 5, part = c >> 6;  // part: which sixteen keys x which 32 values of D
        const int s = part / (D / 32) * 16 + 4 * h, d = part % (D / 32) * 32 + (lane & 31);
        uint32_t p[4];
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const int key = s + (j < 2 ? 2 * j : 8 + 2 * (j - 2));
            p[j] = (uint32_t)tile[key][d] | (uint32_t)tile[key + 1][d] << 16;
        }
        values[block * kChunks + c] = make_uint4(p[0], p[1], p[2], p[3]);
    }
}

// RG row groups of 32 rows a block, 4 / RG wavefronts on each: two wavefronts a SIMD hold 64 accumulators, the query's 32
// operand registers and one tile of keys and values in flight (D = 128).
template <typename T, int D, int RG, int TERMS>
__global__ void __launch_bounds__(64 * kWaves, 2) prompt_attention_kernel(const PromptArgs a) {
    constexpr int KP = kWaves / RG, KS = D / 16, DB = D / 32;
    constexpr int kChunks = kKeys * D / 8;
    constexpr int kStride = D + 4;  // floats of a row of partial outputs: 16-byte aligned, banks shifted row by row
    __shared__ __align__(16) float merge[KP > 1 ? kWaves * kRows * kStride : 4];
    __shared__ float state_m[kWaves][kRows], state_l[kWaves][kRows];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int col = lane & 31, half = lane >> 5;
    const int rg = wave / KP, kp = wave % KP;
    // blocks of one key head lie `heads` apart: on one XCD, whose L2 then holds that head's keys, where heads is a multiple of 8
    const int heads = gridDim.x / ((a.row_tiles + RG - 1) / RG);
    const int head = blockIdx.x % heads, b = (a.head0 + head) / a.key_heads, hk = (a.head0 + head) % a.key_heads;
    const int block_tile = (a.row_tiles + RG - 1) / RG - 1 - blockIdx.x / heads;  // (the longest rows of a causal product first)
    const int rows = a.rep * a.queries, r0 = (block_tile * RG + rg) * kRows, r = r0 + col;
    const bool live = r < rows;
    const int i = live ? r / a.rep : a.queries - 1, h = live ? hk * a.rep + r % a.rep : hk * a.rep;
    const int64_t row = ((int64_t)b * a.query_heads + h) * a.queries + i;
    // the last key a row sees, the last one any and the last one all of this wavefront's rows see
    const int last = a.causal ? a.positions - a.queries + i : a.positions - 1;
    const int any_i = (r0 + kRows - 1 < rows ? r0 + kRows - 1 : rows - 1) / a.rep, all_i = (r0 < rows ? r0 : rows - 1) / a.rep;
    const int any_last = a.causal ? a.positions - a.queries + any_i : a.positions - 1;
    const int all_last = a.causal ? a.positions - a.queries + all_i : a.positions - 1;

    uint4 qf[KS];
#pragma unroll
    for (int s = 0; s < KS; s++) qf[s] = *reinterpret_cast<const uint4 *>((const T *)a.q + row * D + 16 * s + 8 * half);
    floatx16_t o[DB];
#pragma unroll
    for (int d = 0; d < DB; d++)
#pragma unroll
        for (int e = 0; e < 16; e++) o[d][e] = 0.0f;
    float m = -1.0e30f, l = 0.0f;  // (finite: a masked score's weight is exp2(-inf - m) = 0 from the first tile on)
    const float scale = a.scale * kLog2e;

    const int per = (a.tiles + a.splits - 1) / a.splits, t_begin = blockIdx.y * per;
    int t_end = t_begin + per < a.tiles ? t_begin + per : a.tiles;
    if (any_last / kKeys + 1 < t_end) t_end = any_last < 0 ? 0 : any_last / kKeys + 1;
    if (r0 >= rows) t_end = 0;  // (a row group past the end)
    const uint4 *kf = a.keys + (int64_t)head * a.tiles * (TERMS * kChunks) + lane, *vf = a.values + (int64_t)head * a.tiles * kChunks + lane;
    uint4 kt[TERMS * KS], vt[KS];
    auto fetch = [&](const uint4 *from, int t, auto &to) {
        constexpr int n = sizeof(to) / sizeof(uint4);
        const uint4 *p = from + (int64_t)(t < a.tiles ? t : a.tiles - 1) * (n * 64);  // (past the end: read, not used)
#pragma unroll
        for (int s = 0; s < n; s++) to[s] = p[64 * s];
    };
    fetch(kf, t_begin + kp, kt);
    fetch(vf, t_begin + kp, vt);
    for (int t = t_begin + kp; t < t_end; t += KP) {
        floatx16_t s;
#pragma unroll
        for (int e = 0; e < 16; e++) s[e] = 0.0f;
#pragma unroll
        for (int term = TERMS - 1; term >= 0; term--)  // (the small ones first)
#pragma unroll
            for (int k = 0; k < KS; k++) s = Ops<T>::mfma(kt[term * KS + k], qf[k], s);
        fetch(kf, t + KP, kt);
        const int key0 = t * kKeys + 4 * half;  // register e: key 8 (e / 4) + 4 half + e % 4
        if (t * kKeys + kKeys - 1 > all_last) {
#pragma unroll
            for (int e = 0; e < 16; e++) s[e] = key0 + 8 * (e >> 2) + (e & 3) <= last ? s[e] * scale : -INFINITY;
        } else {
#pragma unroll
            for (int e = 0; e < 16; e++) s[e] *= scale;
        }
        float top = s[0];
#pragma unroll
        for (int e = 1; e < 16; e++) top = fmaxf(top, s[e]);
        top = fmaxf(top, __shfl_xor(top, 32));
        // The accumulators are rescaled only when a maximum has grown by more than 2^8: until then the weights are at most
        // 2^8 and their sums stay exact to the same relative error (float32 sums; bfloat16 and float16 hold 2^8).
        if (__any(top > m + 8.0f)) {
            const float m_new = fmaxf(m, top), f = exp2f(m - m_new);
            m = m_new, l *= f;
#pragma unroll
            for (int d = 0; d < DB; d++)
#pragma unroll
                for (int e = 0; e < 16; e++) o[d][e] *= f;
        }
#pragma unroll
        for (int e = 0; e < 16; e++) s[e] = __builtin_amdgcn_exp2f(s[e] - m);
#pragma unroll
        for (int e = 0; e < 16; e++) l += s[e];
        uint4 p[2];
#pragma unroll
        for (int k = 0; k < 2; k++)
            p[k] = make_uint4(Ops<T>::pack(s[8 * k], s[8 * k + 1]), Ops<T>::pack(s[8 * k + 2], s[8 * k + 3]),
                              Ops<T>::pack(s[8 * k + 4], s[8 * k + 5]), Ops<T>::pack(s[8 * k + 6], s[8 * k + 7]));
#pragma unroll
        for (int k = 0; k < 2; k++)
#pragma unroll
            for (int d = 0; d < DB; d++) o[d] = Ops<T>::mfma(vt[k * DB + d], p[k], o[d]);
        fetch(vf, t + KP, vt);
    }
    l += __shfl_xor(l, 32);

    // the wavefronts of a row group: their states brought to one maximum and added up
    if (KP > 1) {
        if (half == 0) state_m[wave][col] = m, state_l[wave][col] = l;
        __syncthreads();
        float top = -1.0e30f, sum = 0.0f;
#pragma unroll
        for (int k = 0; k < KP; k++) top = fmaxf(top, state_m[rg * KP + k][col]);
#pragma unroll
        for (int k = 0; k < KP; k++) sum += state_l[rg * KP + k][col] * exp2f(state_m[rg * KP + k][col] - top);
        const float f = exp2f(m - top);
        float *mine = merge + (wave * kRows + col) * kStride;
#pragma unroll
        for (int d = 0; d < DB; d++)
#pragma unroll
            for (int e = 0; e < 4; e++)
                *reinterpret_cast<float4 *>(mine + 32 * d + 8 * e + 4 * half) =
                    make_float4(o[d][4 * e] * f, o[d][4 * e + 1] * f, o[d][4 * e + 2] * f, o[d][4 * e + 3] * f);
        m = top, l = sum;
        __syncthreads();
    }
    const bool whole = a.splits == 1;
    float inv = 1.0f;
    float *state = nullptr;  // of this row and split: maximum, denominator, weighted sums
    if (whole) {
        float denom = l, f = 1.0f;
        if (a.sinks != nullptr) {
            const float sink = Elem<T>::load((const T *)a.sinks, h) * kLog2e, top = fmaxf(m, sink);
            f = exp2f(m - top), denom = denom * f + exp2f(sink - top);
        }
        inv = f / denom;
    } else {
        state = a.partials + (((int64_t)blockIdx.y * heads + head) * rows + (live ? r : 0)) * (D + 2);
        if (live && kp == 0 && half == 0) state[0] = m, state[1] = l;
    }
    T *out = (T *)a.out + row * D;
#pragma unroll
    for (int d = 0; d < DB; d++)
#pragma unroll
        for (int e = 0; e < 4; e++) {
            if (KP > 1 && (4 * d + e) % KP != kp) continue;
            const int c = 32 * d + 8 * e + 4 * half;
            float4 v;
            if (KP > 1) {
                v = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
#pragma unroll
                for (int k = 0; k < KP; k++) {
                    const float4 w = *reinterpret_cast<const float4 *>(merge + ((rg * KP + k) * kRows + col) * kStride + c);
                    v.x += w.x, v.y += w.y, v.z += w.z, v.w += w.w;
                }
            } else {
                v = make_float4(o[d][4 * e], o[d][4 * e + 1], o[d][4 * e + 2], o[d][4 * e + 3]);
            }
            if (!live) continue;
            if (whole) {
                *reinterpret_cast<uint2 *>(out + c) = make_uint2(Ops<T>::pack(v.x * inv, v.y * inv), Ops<T>::pack(v.z * inv, v.w * inv));
            } else {
                *reinterpret_cast<float2 *>(state + 2 + c) = make_float2(v.x, v.y);
                *reinterpret_cast<float2 *>(state + 4 + c) = make_float2(v.z, v.w);
            }
        }
}

// The splits of a row merged.
template <typename T, int D>
__global__ void __launch_bounds__(kMergeParts * D) prompt_merge_kernel(const PromptArgs a) {
    const int rows = a.rep * a.queries;
    const int64_t all = (int64_t)gridDim.x * gridDim.y;  // rows x (batch x key heads)
    const int r = blockIdx.x, head = blockIdx.y, b = (a.head0 + head) / a.key_heads, hk = (a.head0 + head) % a.key_heads;
    const int h = hk * a.rep + r % a.rep, i = r / a.rep;
    merge_attention_states<T, D>(a.partials + ((int64_t)head * rows + r) * (D + 2), all * (D + 2), a.splits, a.sinks != nullptr,
                                 a.sinks != nullptr ? Elem<T>::load((const T *)a.sinks, h) * kLog2e : 0.0f,
                                 (T *)a.out + (((int64_t)b * a.query_heads + h) * a.queries + i) * D);
}

// The same for few splits, D / 4 threads a row.
template <typename T, int D>
__global__ void __launch_bounds__(256) prompt_merge_few_kernel(const PromptArgs a) {
    const int rows = a.rep * a.queries, r = (int)blockIdx.x * (1024 / D) + (int)threadIdx.x / (D / 4);
    if (r >= rows) return;
    const int head = blockIdx.y, b = (a.head0 + head) / a.key_heads, hk = (a.head0 + head) % a.key_heads;
    const int h = hk * a.rep + r % a.rep, i = r / a.rep;
    merge_few_states<T, D>(a.partials + ((int64_t)head * rows + r) * (D + 2), (int64_t)rows * gridDim.y * (D + 2), a.splits, a.sinks != nullptr,
                           a.sinks != nullptr ? Elem<T>::load((const T *)a.sinks, h) * kLog2e : 0.0f,
                           (T *)a.out + (((int64_t)b * a.query_heads + h) * a.queries + i) * D, (int)threadIdx.x % (D / 4) * 4);
}

struct Plan {
    int tiles, row_tiles, row_groups, splits, terms;
    int64_t heads, slice;  // all (batch, key head)s, and those of one launch
    int64_t rows;
    size_t key_bytes, value_bytes, partial_bytes;
};

// Operands of more heads than this go one slice after the other through one workspace: 32 batches x 8 key heads over 32768 positions
// are 4.3 GB of them.  (256 MB is also what the chip's last cache holds.)
constexpr int64_t kOperandMost = 256LL << 20;

// Whether the composition's product holds keys in float32: outputs of 1024 and more per row, but for bfloat16 products of more than
// 16 rows up to 8192 outputs, which take the CPU's weights as the products of fewer do.
bool keys_are_two_terms(const nvq_attention_prompt_desc &p) {
    return p.cache.positions >= 1024 && !(p.cache.dtype == NVQ_BF16 && p.queries > 16 && p.cache.positions < 8192);
}

// Row groups a block: four (every tile of keys read once per 128 rows) where that gives two blocks per compute unit, else two,
// else one (four wavefronts on the same 32 rows); then, with fewer blocks than compute units still, splits of the keys over the
// grid of at least eight tiles each.
Plan prompt_plan(const nvq_attention_prompt_desc &p) {
    const nvq_attention_desc &d = p.cache;
    Plan r{};
    r.heads = d.batch * d.key_heads;
    r.rows = d.query_heads / d.key_heads * p.queries;
    r.tiles = (int)((d.positions + kKeys - 1) / kKeys);
    r.row_tiles = (int)((r.rows + kRows - 1) / kRows);
    r.terms = keys_are_two_terms(p) ? 2 : 1;
    const int64_t head_bytes = (int64_t)r.tiles * kKeys * d.head_dim * 2, most = kOperandMost / ((r.terms + 1) * head_bytes);
    const int64_t slices = (r.heads + (most > 1 ? most : 1) - 1) / (most > 1 ? most : 1);
    r.slice = slices > 1 ? (r.heads + slices - 1) / slices : r.heads;
    const int64_t cus = compute_units();
    r.row_groups = 1;
    for (int g = 4; g > 1; g /= 2)
        if (r.slice * ((r.row_tiles + g - 1) / g) >= 2 * cus) {
            r.row_groups = g;
            break;
        }
    r.splits = 1;
    const int64_t blocks = r.slice * r.row_tiles;
    if (r.row_groups == 1 && blocks < cus && blocks > 0) {
        int64_t want = (2 * cus + blocks - 1) / blocks;
        if (want > r.tiles / 8) want = r.tiles / 8;
        if (want > 32) want = 32;
        if (want > 1) {
            const int64_t per = (r.tiles + want - 1) / want;
            r.splits = (int)((r.tiles + per - 1) / per);
        }
    }
    r.key_bytes = (size_t)(r.slice * r.terms * head_bytes), r.value_bytes = (size_t)(r.slice * head_bytes);
    r.partial_bytes = r.splits > 1 ? (size_t)r.splits * r.slice * r.rows * (d.head_dim + 2) * sizeof(float) : 0;
    return r;
}

template <typename T, int D, int TERMS>
int32_t run_rows(const PromptArgs &a, const Plan &p, int64_t heads, hipStream_t s) {
    const dim3 grid((unsigned)(heads * ((p.row_tiles + p.row_groups - 1) / p.row_groups)), (unsigned)p.splits), block(64 * kWaves);
    switch (p.row_groups) {
    case 4: hipLaunchKernelGGL((prompt_attention_kernel<T, D, 4, TERMS>), grid, block, 0, s, a); break;
    case 2: hipLaunchKernelGGL((prompt_attention_kernel<T, D, 2, TERMS>), grid, block, 0, s, a); break;
    default: hipLaunchKernelGGL((prompt_attention_kernel<T, D, 1, TERMS>), grid, block, 0, s, a); break;
    }
    NVQ_LAUNCH_CHECK("quantized_attention");
    if (p.splits > 1) {
        const unsigned blocks = (unsigned)((p.rows + 1024 / D - 1) / (1024 / D));  // (of 256 threads, few splits)
        if (p.splits <= kFewSplits) hipLaunchKernelGGL((prompt_merge_few_kernel<T, D>), dim3(blocks, (unsigned)heads), dim3(256), 0, s, a);
        else hipLaunchKernelGGL((prompt_merge_kernel<T, D>), dim3((unsigned)p.rows, (unsigned)heads), dim3(kMergeParts * D), 0, s, a);
        NVQ_LAUNCH_CHECK("quantized_attention merge");
    }
    return NVQ_OK;
}

template <typename T, int D, int TERMS>
int32_t run_sized(const nvq_attention_prompt_desc &desc, const Plan &p, const void *q, const void *kw, const void *ks, const void *kb,
                  const void *vw, const void *vs, const void *vb, const void *sinks, void *out, void *workspace, hipStream_t s) {
    const nvq_attention_desc &d = desc.cache;
    uint4 *keys = (uint4 *)workspace, *values = keys + p.key_bytes / 16;
    int shift = 5;
    while ((1 << shift) < d.group_size) shift++;
    PromptArgs a{};
    a.q = q, a.keys = keys, a.values = values, a.sinks = sinks, a.out = out;
    a.partials = (float *)((char *)workspace + p.key_bytes + p.value_bytes);
    a.scale = d.scale, a.causal = desc.causal;
    a.query_heads = (int)d.query_heads, a.key_heads = (int)d.key_heads, a.rep = (int)(d.query_heads / d.key_heads);
    a.queries = (int)desc.queries, a.positions = (int)d.positions;
    a.tiles = p.tiles, a.row_tiles = p.row_tiles, a.splits = p.splits;
    for (int64_t first = 0; first < p.heads; first += p.slice) {  // (the stream keeps a slice's readers ahead of the next one's writers)
        const int64_t heads = p.heads - first < p.slice ? p.heads - first : p.slice;
        const dim3 grid((unsigned)p.tiles, (unsigned)heads);
        a.head0 = (int)first;
#define NVQ_OPERANDS(B)                                                                                                                             case B:                                                                                                                                             hipLaunchKernelGGL((prompt_operands_kernel<T, B, D, TERMS>), grid, dim3(256), 0, s, (const uint32_t *)kw, (const T *)ks, (const T *)kb,                            (const uint32_t *)vw, (const T *)vs, (const T *)vb, a.head0, (int)d.positions, shift, keys, values);                          break;
        switch (d.bits) { NVQ_OPERANDS(1) NVQ_OPERANDS(2) NVQ_OPERANDS(3) NVQ_OPERANDS(4) NVQ_OPERANDS(5) NVQ_OPERANDS(6) NVQ_OPERANDS(8) }
#undef NVQ_OPERANDS
        NVQ_LAUNCH_CHECK("quantized_attention operands");
        const int32_t rc = run_rows<T, D, TERMS>(a, p, heads, s);
        if (rc != NVQ_OK) return rc;
    }
    return NVQ_OK;
}

template <typename T, typename... A>
int32_t run_type(const nvq_attention_prompt_desc &d, A... args) {
    const Plan p = prompt_plan(d);
    if (d.cache.head_dim == 64) return p.terms == 2 ? run_sized<T, 64, 2>(d, p, args...) : run_sized<T, 64, 1>(d, p, args...);
    return p.terms == 2 ? run_sized<T, 128, 2>(d, p, args...) : run_sized<T, 128, 1>(d, p, args...);
}

}  // namespace

size_t attention_prompt_workspace_bytes(const nvq_attention_prompt_desc &d) {
    const Plan p = prompt_plan(d);
    return p.key_bytes + p.value_bytes + p.partial_bytes;
}

int32_t launch_attention_prompt(const nvq_attention_prompt_desc &d, const void *q, const void *kw, const void *ks, const void *kb,
                                const void *vw, const void *vs, const void *vb, const void *sinks, void *out, void *workspace, hipStream_t s) {
    return d.cache.dtype == NVQ_BF16 ? run_type<bf16_t>(d, q, kw, ks, kb, vw, vs, vb, sinks, out, workspace, s)
                                     : run_type<f16_t>(d, q, kw, ks, kb, vw, vs, vb, sinks, out, workspace, s);
}

}  // namespace nvq
