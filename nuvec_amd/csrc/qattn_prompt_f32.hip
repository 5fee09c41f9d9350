// Attention of several query rows per head over an affine-quantized key / value cache in float32 (reference:
// crates/nuvec-core/src/fast/imp.rs:3996-4035, the composition of two quantized products and a softmax; nuvec-lm's causal mask,
// crates/nuvec-lm/src/model.rs:3646-3700):
//     out[b, h, i, :] = softmax(scale * q[b, h, i, :] . K[b, h / rep]^T [masked] [, sink[h]]) . V[b, h / rep]
// with keys, values, scores and weights in float32 throughout, keys and values as nuvec's CPU product dequantizes them (two roundings,
// crates/nuvec-core/src/kernels.rs:835-859), and the scores never in memory.
//
// The rows of a key head are its rep x L query rows (row r: query r / rep, head r % rep).  A wavefront owns 32 rows, two tiles of
// sixteen, and takes 32 keys at a time on v_mfma_f32_16x16x4_f32, scores transposed: S^T = K . Q^T.  The contraction's order is free,
// so lane (quarter q, key l) takes the values D / 4 q .. of its key, whole runs of codes straight from the cache, and the queries lie
// the same way in registers; the scores come with a lane's four keys beside each other, which is the operand O^T = V^T . P^T wants.
// V is dequantized the same way and turned through a piece of LDS of the wavefront's own.
//
// What fills the chip: few rows are walked by four wavefronts of a block, each taking every fourth tile of keys, and where that leaves
// compute units idle by several blocks whose float32 states a second kernel merges.
//
// Bound by the float32 matrix instruction (32 of 16 x 16 x 4 a tile of 32 keys and head size 64, a microsecond) and the dequantization
// beside it; the composition ran both products on the vector kernels, four rows a pass over the cache.  us and error against float64,
// composition -> here, causal: 281 queries of 4 x 4 heads over 284 positions, D = 64, 509 -> 21, 4.9e-7 -> 1.7e-7; 34 queries of 8 x 4
// heads over 1218 positions, D = 128, 541 -> 31, 9.5e-7 -> 2.8e-7; 2 queries of 8 heads over 8192 positions 118 -> 20.
#include "attention_merge.h"
#include "nvq_device.h"
#include "nvq_internal.h"
#include "qmf_kernel.h"

#include <float.h>

namespace nvq {
namespace {

using qmf::static_for;

typedef float f32x4_t __attribute__((ext_vector_type(4)));

constexpr int kKeys = 32;   // keys of a tile, in two halves of sixteen
constexpr int kRows = 32;   // rows of a wavefront, likewise
constexpr int kWaves = 4;   // of a block: row groups x parts of the keys

struct Args {
    const float *q;
    const uint32_t *kw, *vw;
    const float *ks, *kb, *vs, *vb, *sinks;
    float *out, *partials;  // states [splits][heads][rows][D + 2]
    float scale, scale_rest;  // of the scores, times log2 e, and what that rounding left
    int32_t causal, query_heads, key_heads, rep, queries, positions, group_shift;
    int32_t tiles, row_tiles, splits;
};

// The D / 4 codes of a lane's part of a row, in dwords from the part's first code on.
template <int BITS, int D>
struct Part {
    static constexpr int kCodes = D / 4, kRowWords = D * BITS / 32;
    static constexpr int kWords = (kCodes * BITS + 31) / 32, kLoads = D == 64 && BITS % 2 != 0 ? kWords + 1 : kWords;
    uint32_t w[kLoads];
    float s, b;
};
template <int BITS, int D>
__device__ __forceinline__ void load_part(const uint32_t *w, const float *s, const float *b, int64_t row, int q, int group_shift, Part<BITS, D> &p) {
    using P = Part<BITS, D>;
    const int first = q * P::kCodes * BITS / 32;  // (an odd width of head size 64 starts in the middle of a dword in odd quarters)
#pragma unroll
    for (int i = 0; i < P::kLoads; i++) p.w[i] = w[row * P::kRowWords + (first + i < P::kRowWords ? first + i : P::kRowWords - 1)];
    const int64_t g = row * (D >> group_shift) + ((q * P::kCodes) >> group_shift);
    p.s = s[g], p.b = b[g];
}
template <int BITS, int D>
__device__ __forceinline__ void dequantize_part(const Part<BITS, D> &p, int q, float (&v)[D / 4]) {
    using P = Part<BITS, D>;
    uint32_t u[P::kWords];
#pragma unroll
    for (int i = 0; i < P::kWords; i++) {
        if constexpr (D == 64 && BITS % 2 != 0) u[i] = __builtin_amdgcn_alignbit(p.w[i + 1], p.w[i], 16 * (q & 1));
        else u[i] = p.w[i];
    }
    static_for<D / 4>([&](auto i_tag) {
        constexpr int i = decltype(i_tag)::value, at = i * BITS / 32, sh = i * BITS % 32;
        uint32_t c = u[at] >> sh;
        if constexpr (sh + BITS > 32) c |= u[at + 1] << (32 - sh);
        v[i] = (float)(c & ((1u << BITS) - 1u)) * p.s + p.b;
    });
}

// RG row groups of 32 rows a block, 4 / RG wavefronts on each.
template <int BITS, int D, int RG>
__global__ void __launch_bounds__(64 * kWaves) __attribute__((amdgpu_waves_per_eu(2, 2))) prompt_attention_f32_kernel(const Args a) {
    constexpr int KP = kWaves / RG, kPart = D / 4, kTiles = D / 16;
    constexpr int kStride = D + 4;  // floats: sixteen lanes of four quarters, or of sixteen rows, fall on all banks
    __shared__ __align__(16) float lds[kWaves][kKeys * kStride];
    __shared__ float state_m[kWaves][kRows], state_l[kWaves][kRows];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int l = lane & 15, q = lane >> 4;
    const int rg = wave / KP, kp = wave % KP;
    const int heads = gridDim.x / ((a.row_tiles + RG - 1) / RG);
    const int head = blockIdx.x % heads, b = head / a.key_heads, hk = head % a.key_heads;
    const int block_tile = (a.row_tiles + RG - 1) / RG - 1 - blockIdx.x / heads;  // (the longest rows of a causal product first)
    const int rows = a.rep * a.queries, r0 = (block_tile * RG + rg) * kRows;
    float *mine = lds[wave];

    // Row l of either tile: its query, and the last key it sees.
    int64_t out_row[2];
    int last[2];
    bool live[2];
    float qf[2][kPart];
#pragma unroll
    for (int t = 0; t < 2; t++) {
        const int r = r0 + 16 * t + l;
        live[t] = r < rows;
        const int i = live[t] ? r / a.rep : a.queries - 1, h = live[t] ? hk * a.rep + r % a.rep : hk * a.rep;
        out_row[t] = ((int64_t)b * a.query_heads + h) * a.queries + i;
        last[t] = a.causal ? a.positions - a.queries + i : a.positions - 1;
        const float4 *from = reinterpret_cast<const float4 *>(a.q + out_row[t] * D + q * kPart);
#pragma unroll
        for (int c = 0; c < kPart / 4; c++) {
            const float4 v = from[c];
            qf[t][4 * c] = v.x, qf[t][4 * c + 1] = v.y, qf[t][4 * c + 2] = v.z, qf[t][4 * c + 3] = v.w;
        }
    }
    const int any_i = (r0 + kRows - 1 < rows ? r0 + kRows - 1 : rows - 1) / a.rep, all_i = (r0 < rows ? r0 : rows - 1) / a.rep;
    const int any_last = a.causal ? a.positions - a.queries + any_i : a.positions - 1;
    const int all_last = a.causal ? a.positions - a.queries + all_i : a.positions - 1;
    const int per = (a.tiles + a.splits - 1) / a.splits, t_begin = blockIdx.y * per;
    int t_end = t_begin + per < a.tiles ? t_begin + per : a.tiles;
    if (any_last / kKeys + 1 < t_end) t_end = any_last < 0 ? 0 : any_last / kKeys + 1;
    if (r0 >= rows) t_end = 0;  // (a row group past the end)

    f32x4_t o[2][kTiles];
#pragma unroll
    for (int t = 0; t < 2; t++)
#pragma unroll
        for (int d = 0; d < kTiles; d++) o[t][d] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
    float m[2] = {-FLT_MAX, -FLT_MAX}, sum[2] = {0.0f, 0.0f};  // (finite: a masked score's weight is exp2(-inf - m) = 0 from the first tile on)

    const int64_t row0 = (int64_t)head * a.positions;
    Part<BITS, D> kc[2], vc[2];
    auto fetch = [&](const uint32_t *w, const float *s, const float *bias, int tile, Part<BITS, D> (&to)[2]) __attribute__((always_inline)) {
#pragma unroll
        for (int t = 0; t < 2; t++) {
            const int key = tile * kKeys + 16 * t + l;  // (past the end: the last one, masked)
            load_part<BITS, D>(w, s, bias, row0 + (key < a.positions ? key : a.positions - 1), q, a.group_shift, to[t]);
        }
    };
    fetch(a.kw, a.ks, a.kb, t_begin + kp, kc);
    fetch(a.vw, a.vs, a.vb, t_begin + kp, vc);
    for (int tile = t_begin + kp; tile < t_end; tile += KP) {
        f32x4_t s[2][2];  // [keys][rows]: element e is key 4 q + e
#pragma unroll
        for (int t = 0; t < 2; t++) {
            float k[kPart];
            dequantize_part<BITS, D>(kc[t], q, k);
            f32x4_t part[2][2];  // (two chains a tile)
#pragma unroll
            for (int c = 0; c < 2; c++) part[c][0] = part[c][1] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
            for (int i = 0; i < kPart; i++)
#pragma unroll
                for (int r = 0; r < 2; r++) part[i & 1][r] = __builtin_amdgcn_mfma_f32_16x16x4f32(k[i], qf[r][i], part[i & 1][r], 0, 0, 0);
#pragma unroll
            for (int r = 0; r < 2; r++) s[t][r] = part[0][r] + part[1][r];
        }
        fetch(a.kw, a.ks, a.kb, tile + KP, kc);
        // V through LDS: row `key` of D values
#pragma unroll
        for (int t = 0; t < 2; t++) {
            float v[kPart];
            dequantize_part<BITS, D>(vc[t], q, v);
#pragma unroll
            for (int c = 0; c < kPart / 4; c++)
                *reinterpret_cast<float4 *>(mine + (16 * t + l) * kStride + q * kPart + 4 * c) = make_float4(v[4 * c], v[4 * c + 1], v[4 * c + 2], v[4 * c + 3]);
        }
        fetch(a.vw, a.vs, a.vb, tile + KP, vc);
        const int key0 = tile * kKeys + 4 * q;
        const bool masked = tile * kKeys + kKeys - 1 > all_last;
#pragma unroll
        for (int r = 0; r < 2; r++) {
            float top = -INFINITY, low = INFINITY;
#pragma unroll
            for (int t = 0; t < 2; t++)
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    if (masked && key0 + 16 * t + e > last[r]) s[t][r][e] = -INFINITY;
                    top = fmaxf(top, s[t][r][e] * a.scale), low = fminf(low, s[t][r][e] * a.scale);
                }
            if (masked) low = -INFINITY;  // (the general form)
            if (a.scale < 0.0f && masked) {  // (a hidden score is the least one whatever the scale's sign)
                top = -INFINITY;
#pragma unroll
                for (int t = 0; t < 2; t++)
#pragma unroll
                    for (int e = 0; e < 4; e++)
                        if (key0 + 16 * t + e <= last[r]) top = fmaxf(top, s[t][r][e] * a.scale);
            }
            top = fmaxf(top, __shfl_xor(top, 16));
            top = fmaxf(top, __shfl_xor(top, 32));
            // (rescaled only when a maximum has grown by more than 2^8: until then the weights are at most 2^8)
            if (__any(top > m[r] + 8.0f)) {
                const float m_new = fmaxf(m[r], top), f = exp2f(m[r] - m_new);
                m[r] = m_new, sum[r] *= f;
#pragma unroll
                for (int d = 0; d < kTiles; d++)
#pragma unroll
                    for (int e = 0; e < 4; e++) o[r][d][e] *= f;
            }
            // Two kinds of scores do not take the exact form below: -inf, which would meet an infinity of either sign, and, as m is a rounded
            // product and they are not, those so large that what the rounding leaves, up to 2^-24 m, is no small power of two.
            if (__any(fabsf(m[r]) > 1048576.0f || low == -INFINITY)) {
#pragma unroll
                for (int t = 0; t < 2; t++)
#pragma unroll
                    for (int e = 0; e < 4; e++) {
                        const bool hidden = masked && key0 + 16 * t + e > last[r];
                        const float v = s[t][r][e] * a.scale, x = __builtin_fmaf(s[t][r][e], a.scale, __builtin_fmaf(s[t][r][e], a.scale_rest, -m[r]));
                        s[t][r][e] = hidden ? 0.0f : __builtin_amdgcn_exp2f(fabsf(m[r]) > 1048576.0f || v == -INFINITY ? v - m[r] : x);
                    }
            } else {
#pragma unroll
                for (int t = 0; t < 2; t++)
#pragma unroll
                    for (int e = 0; e < 4; e++)
                        s[t][r][e] = __builtin_amdgcn_exp2f(__builtin_fmaf(s[t][r][e], a.scale, __builtin_fmaf(s[t][r][e], a.scale_rest, -m[r])));
            }
#pragma unroll
            for (int t = 0; t < 2; t++) sum[r] += (s[t][r][0] + s[t][r][1]) + (s[t][r][2] + s[t][r][3]);
        }
        __builtin_amdgcn_wave_barrier();  // (the wavefront's LDS accesses execute in order)
#pragma unroll
        for (int t = 0; t < 2; t++)
#pragma unroll
            for (int e = 0; e < 4; e++)
#pragma unroll
                for (int d = 0; d < kTiles; d++) {
                    const float v = mine[(16 * t + 4 * q + e) * kStride + 16 * d + l];
#pragma unroll
                    for (int r = 0; r < 2; r++) o[r][d] = __builtin_amdgcn_mfma_f32_16x16x4f32(v, s[t][r][e], o[r][d], 0, 0, 0);
                }
        __builtin_amdgcn_wave_barrier();
    }
#pragma unroll
    for (int r = 0; r < 2; r++) {
        sum[r] += __shfl_xor(sum[r], 16);
        sum[r] += __shfl_xor(sum[r], 32);
    }

    // The wavefronts of a row group: their states brought to one maximum and added up, row 16 r + l by lane (q, l)'s quarters.
    if (KP > 1) {
#pragma unroll
        for (int r = 0; r < 2; r++)
            if (q == 0) state_m[wave][16 * r + l] = m[r], state_l[wave][16 * r + l] = sum[r];
        __syncthreads();
#pragma unroll
        for (int r = 0; r < 2; r++) {
            float top = -FLT_MAX, all = 0.0f;
#pragma unroll
            for (int k = 0; k < KP; k++) top = fmaxf(top, state_m[rg * KP + k][16 * r + l]);
#pragma unroll
            for (int k = 0; k < KP; k++) all += state_l[rg * KP + k][16 * r + l] * exp2f(state_m[rg * KP + k][16 * r + l] - top);
            const float f = exp2f(m[r] - top);
#pragma unroll
            for (int d = 0; d < kTiles; d++)
                *reinterpret_cast<float4 *>(mine + (16 * r + l) * kStride + 16 * d + 4 * q) = make_float4(o[r][d][0] * f, o[r][d][1] * f, o[r][d][2] * f, o[r][d][3] * f);
            m[r] = top, sum[r] = all;
        }
        __syncthreads();
    }
#pragma unroll
    for (int r = 0; r < 2; r++) {
        if (!live[r]) continue;
        float inv = 1.0f;
        float *state = nullptr;
        if (a.splits == 1) {
            float denom = sum[r], f = 1.0f;
            if (a.sinks != nullptr) {
                const int h = (int)(out_row[r] / a.queries % a.query_heads);
                const float sink = a.sinks[h] * 1.44269504088896340736f, top = fmaxf(m[r], sink);
                f = exp2f(m[r] - top), denom = denom * f + exp2f(sink - top);
            }
            inv = f / denom;
        } else {
            state = a.partials + (((int64_t)blockIdx.y * heads + head) * rows + r0 + 16 * r + l) * (D + 2);
            if (kp == 0 && q == 0) state[0] = m[r], state[1] = sum[r];
        }
#pragma unroll
        for (int d = 0; d < kTiles; d++) {
            if (KP > 1 && d % KP != kp) continue;
            float4 v = make_float4(o[r][d][0], o[r][d][1], o[r][d][2], o[r][d][3]);
            if (KP > 1) {
                v = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
#pragma unroll
                for (int k = 0; k < KP; k++) {
                    const float4 w = *reinterpret_cast<const float4 *>(lds[rg * KP + k] + (16 * r + l) * kStride + 16 * d + 4 * q);
                    v.x += w.x, v.y += w.y, v.z += w.z, v.w += w.w;
                }
            }
            if (a.splits == 1) {
                *reinterpret_cast<float4 *>(a.out + out_row[r] * D + 16 * d + 4 * q) = make_float4(v.x * inv, v.y * inv, v.z * inv, v.w * inv);
            } else {
                *reinterpret_cast<float2 *>(state + 2 + 16 * d + 4 * q) = make_float2(v.x, v.y);
                *reinterpret_cast<float2 *>(state + 4 + 16 * d + 4 * q) = make_float2(v.z, v.w);
            }
        }
    }
}

// The splits of a row merged.
template <int D>
__global__ void __launch_bounds__(kMergeParts * D) prompt_merge_f32_kernel(const Args a) {
    const int rows = a.rep * a.queries;
    const int64_t all = (int64_t)gridDim.x * gridDim.y;  // rows x heads
    const int r = blockIdx.x, head = blockIdx.y, b = head / a.key_heads, hk = head % a.key_heads;
    const int h = hk * a.rep + r % a.rep, i = r / a.rep;
    merge_attention_states<float, D>(a.partials + ((int64_t)head * rows + r) * (D + 2), all * (D + 2), a.splits, a.sinks != nullptr,
                                     a.sinks != nullptr ? a.sinks[h] * 1.44269504088896340736f : 0.0f,
                                     a.out + (((int64_t)b * a.query_heads + h) * a.queries + i) * D);
}

// The same for few splits, D / 4 threads a row.
template <int D>
__global__ void __launch_bounds__(256) prompt_merge_few_f32_kernel(const Args a) {
    const int rows = a.rep * a.queries, r = (int)blockIdx.x * (1024 / D) + (int)threadIdx.x / (D / 4);
    if (r >= rows) return;
    const int head = blockIdx.y, b = head / a.key_heads, hk = head % a.key_heads;
    const int h = hk * a.rep + r % a.rep, i = r / a.rep;
    merge_few_states<float, D>(a.partials + ((int64_t)head * rows + r) * (D + 2), (int64_t)rows * gridDim.y * (D + 2), a.splits, a.sinks != nullptr,
                               a.sinks != nullptr ? a.sinks[h] * 1.44269504088896340736f : 0.0f,
                               a.out + (((int64_t)b * a.query_heads + h) * a.queries + i) * D, (int)threadIdx.x % (D / 4) * 4);
}

struct Plan { int tiles, row_tiles, row_groups, splits; int64_t heads, rows; };

// Four row groups a block where that gives two blocks a compute unit; else four wavefronts on each, and with fewer than two blocks a
// unit splits of the keys over the grid, of a tile a wavefront at least.
Plan plan_of(const nvq_attention_prompt_desc &p) {
    const nvq_attention_desc &d = p.cache;
    Plan r{};
    r.heads = d.batch * d.key_heads;
    r.rows = d.query_heads / d.key_heads * p.queries;
    r.tiles = (int)((d.positions + kKeys - 1) / kKeys);
    r.row_tiles = (int)((r.rows + kRows - 1) / kRows);
    const int64_t cus = compute_units(), blocks = r.heads * r.row_tiles;
    r.row_groups = r.heads * ((r.row_tiles + 3) / 4) >= 2 * cus ? 4 : 1;
    r.splits = 1;
    if (r.row_groups == 1 && blocks < 2 * cus && blocks > 0) {
        int64_t want = (2 * cus + blocks - 1) / blocks;
        if (want > r.tiles / 4) want = r.tiles / 4;
        if (want > 32) want = 32;
        if (want > 1) {
            const int64_t per = (r.tiles + want - 1) / want;
            r.splits = (int)((r.tiles + per - 1) / per);
        }
    }
    return r;
}

template <int BITS, int D>
int32_t run(const Args &a, const Plan &p, hipStream_t s) {
    const dim3 grid((unsigned)(p.heads * ((p.row_tiles + p.row_groups - 1) / p.row_groups)), (unsigned)p.splits), block(64 * kWaves);
    if (p.row_groups == 4) hipLaunchKernelGGL((prompt_attention_f32_kernel<BITS, D, 4>), grid, block, 0, s, a);
    else hipLaunchKernelGGL((prompt_attention_f32_kernel<BITS, D, 1>), grid, block, 0, s, a);
    NVQ_LAUNCH_CHECK("quantized_attention");
    if (p.splits > 1) {
        const unsigned blocks = (unsigned)((p.rows + 1024 / D - 1) / (1024 / D));  // (of 256 threads, few splits)
        if (p.splits <= kFewSplits) hipLaunchKernelGGL((prompt_merge_few_f32_kernel<D>), dim3(blocks, (unsigned)p.heads), dim3(256), 0, s, a);
        else hipLaunchKernelGGL((prompt_merge_f32_kernel<D>), dim3((unsigned)p.rows, (unsigned)p.heads), dim3(kMergeParts * D), 0, s, a);
        NVQ_LAUNCH_CHECK("quantized_attention merge");
    }
    return NVQ_OK;
}

template <int BITS>
int32_t run_sized(const Args &a, const Plan &p, int head_dim, hipStream_t s) { return head_dim == 64 ? run<BITS, 64>(a, p, s) : run<BITS, 128>(a, p, s); }

}  // namespace

size_t attention_prompt_f32_workspace_bytes(const nvq_attention_prompt_desc &d) {
    const Plan p = plan_of(d);
    return p.splits > 1 ? (size_t)p.splits * p.heads * p.rows * (d.cache.head_dim + 2) * sizeof(float) : 0;
}

int32_t launch_attention_prompt_f32(const nvq_attention_prompt_desc &desc, const void *q, const void *kw, const void *ks, const void *kb,
                                    const void *vw, const void *vs, const void *vb, const void *sinks, void *out, void *workspace, hipStream_t s) {
    const nvq_attention_desc &d = desc.cache;
    const Plan p = plan_of(desc);
    int shift = 5;
    while ((1 << shift) < d.group_size) shift++;
    const double scale = (double)d.scale * 1.44269504088896340736;
    Args a{};
    a.q = (const float *)q, a.kw = (const uint32_t *)kw, a.vw = (const uint32_t *)vw, a.ks = (const float *)ks, a.kb = (const float *)kb;
    a.vs = (const float *)vs, a.vb = (const float *)vb, a.sinks = (const float *)sinks, a.out = (float *)out, a.partials = (float *)workspace;
    a.scale = (float)scale, a.scale_rest = (float)(scale - (double)a.scale), a.causal = desc.causal;
    a.query_heads = (int)d.query_heads, a.key_heads = (int)d.key_heads, a.rep = (int)(d.query_heads / d.key_heads);
    a.queries = (int)desc.queries, a.positions = (int)d.positions, a.group_shift = shift;
    a.tiles = p.tiles, a.row_tiles = p.row_tiles, a.splits = p.splits;
    switch (d.bits) {
    case 1: return run_sized<1>(a, p, d.head_dim, s);
    case 2: return run_sized<2>(a, p, d.head_dim, s);
    case 3: return run_sized<3>(a, p, d.head_dim, s);
    case 4: return run_sized<4>(a, p, d.head_dim, s);
    case 5: return run_sized<5>(a, p, d.head_dim, s);
    case 6: return run_sized<6>(a, p, d.head_dim, s);
    default: return run_sized<8>(a, p, d.head_dim, s);
    }
}

}  // namespace nvq
