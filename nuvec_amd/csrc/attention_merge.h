// The states that the splits of a row's positions leave (maximum of the base-2 scores, denominator, D weighted sums, all
// float32) merged into the row's output, optionally with an attention sink.
//
// Bound by the round trips to the states: one thread per value that walked the splits one after the other, twice, took most
// of the pass (2 x 2 key heads over 19720 positions of 8-bit codes in 64 splits: 46 us, with this merge 21; 341 queries of 2
// heads over 7868 positions 29 -> 19).  Here lane z of every wavefront holds split z's
// weight (at most 64 splits), four groups of D threads take the splits in turn, eight loads under way at a time, and add up
// through LDS.
#pragma once

#include "nvq_device.h"

#include <float.h>

namespace nvq {

constexpr int kMergeParts = 4;

// Block: kMergeParts x D threads, one row.  `src` is the row's first state, `stride` floats lie between the states of
// consecutive splits; `sink` is in base 2.
template <typename T, int D>
__device__ __forceinline__ void merge_attention_states(const float *__restrict__ src, int64_t stride, int splits, bool has_sink, float sink,
                                                       T *__restrict__ out) {
    __shared__ float part[kMergeParts][D];
    const int lane = threadIdx.x & 63, at = threadIdx.x % D, group = threadIdx.x / D;
    const bool real = lane < splits;
    const float m = real ? src[lane * stride] : -FLT_MAX, l = real ? src[lane * stride + 1] : 0.0f;
    float top = m;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) top = fmaxf(top, __shfl_xor(top, o));
    if (has_sink) top = fmaxf(top, sink);
    const float w = real ? exp2f(m - top) : 0.0f;
    float denom = l * w, sum = 0.0f;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) denom += __shfl_xor(denom, o);
    if (has_sink) denom += exp2f(sink - top);
    for (int z0 = group; z0 < splits; z0 += 8 * kMergeParts) {  // (uniform in a wavefront: D is 64 or 128)
        float v[8];
#pragma unroll
        for (int i = 0; i < 8; i++) {
            const int z = z0 + kMergeParts * i;
            v[i] = src[(z < splits ? z : splits - 1) * stride + 2 + at];
        }
#pragma unroll
        for (int i = 0; i < 8; i++) {
            const int z = z0 + kMergeParts * i;
            if (z < splits) sum = __builtin_fmaf(v[i], __shfl(w, z), sum);
        }
    }
    part[group][at] = sum;
    __syncthreads();
    if (group != 0) return;
    sum = (part[0][at] + part[1][at]) + (part[2][at] + part[3][at]);
    Elem<T>::store(out, at, sum / denom);
}

// Up to eight splits: a row is D / 4 threads, each with four values of all splits under way at once; the sums are those of
// merge_attention_states, in its order, without its shuffles, LDS and wait.  A block a row cost 6192 rows of two splits (129 queries of
// 16 heads x 3 over 536 positions of 8 bits) half of the call: 34.6 us there, 23.1 here; 284 queries of 16 heads over 4873 positions
// 53 -> 45; 16 x 32 rows of one query over 8192 positions 41.7 -> 40.1.
constexpr int kFewSplits = 8;
template <typename T, int D>
__device__ __forceinline__ void merge_few_states(const float *__restrict__ src, int64_t stride, int splits, bool has_sink, float sink, T *__restrict__ out,
                                                 int at) {
    float m[kFewSplits], l[kFewSplits], v[kFewSplits][4];
#pragma unroll
    for (int z = 0; z < kFewSplits; z++) {
        const float *state = src + (z < splits ? z : 0) * stride;
        const float2 head = *reinterpret_cast<const float2 *>(state);
        const float2 a = *reinterpret_cast<const float2 *>(state + 2 + at), b = *reinterpret_cast<const float2 *>(state + 4 + at);
        m[z] = z < splits ? head.x : -FLT_MAX, l[z] = z < splits ? head.y : 0.0f;
        v[z][0] = a.x, v[z][1] = a.y, v[z][2] = b.x, v[z][3] = b.y;
    }
    float top = m[0];
#pragma unroll
    for (int z = 1; z < kFewSplits; z++) top = fmaxf(top, m[z]);
    if (has_sink) top = fmaxf(top, sink);
    float w[kFewSplits];
#pragma unroll
    for (int z = 0; z < kFewSplits; z++) w[z] = z < splits ? exp2f(m[z] - top) : 0.0f, l[z] *= w[z];
    float denom = ((l[0] + l[1]) + (l[2] + l[3])) + ((l[4] + l[5]) + (l[6] + l[7]));
    if (has_sink) denom += exp2f(sink - top);
#pragma unroll
    for (int i = 0; i < 4; i++) {
        float part[kMergeParts];
#pragma unroll
        for (int g = 0; g < kMergeParts; g++) {
            part[g] = g < splits ? __builtin_fmaf(v[g][i], w[g], 0.0f) : 0.0f;
            if (g + kMergeParts < splits) part[g] = __builtin_fmaf(v[g + kMergeParts][i], w[g + kMergeParts], part[g]);
        }
        Elem<T>::store(out, at + i, ((part[0] + part[1]) + (part[2] + part[3])) / denom);
    }
}

}  // namespace nvq
