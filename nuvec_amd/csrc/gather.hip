// Index helpers of the gathered products (reference: crates/nuvec-core/src/kernels.rs:873-892,
// crates/nuvec-kernels/src/metal/gather_gemm.metal:436-457).
#include "nvq_device.h"
#include "nvq_internal.h"
#include "wave_reduce.h"

namespace nvq {
namespace {

// offsets[row, g] = first position of `indices[row, :]` whose value is not below g
// (a lower bound by binary search; the row is sorted by the caller's contract).
__global__ void sorted_offsets_kernel(const uint32_t *__restrict__ indices, int64_t rows, int64_t m, int32_t groups,
                                      int32_t *__restrict__ offsets) {
    const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= rows * groups) return;
    const int64_t r = t / groups;
    const uint32_t g = (uint32_t)(t % groups);
    const uint32_t *row = indices + r * m;
    int64_t lo = 0, hi = m;
    while (lo < hi) {
        const int64_t mid = lo + (hi - lo) / 2;
        if (row[mid] < g) lo = mid + 1; else hi = mid;
    }
    offsets[t] = (int32_t)lo;
}

// The pairs (token, choice) of a mixture-of-experts layer ordered by expert, stably: what SwitchGlu::forward gets
// from `argsort` of the flattened expert ids, its inverse, and `sorted_offsets` of the sorted ids
// (crates/nuvec-lm/src/model.rs:2193-2210), in one block.  A counting sort: a histogram of the ids in LDS, an
// exclusive scan over the experts (the offsets), then the pairs placed chunk by chunk in pair order; inside a
// chunk a pair's rank among the equal ids before it comes from wavefront ballots (lanes before it in its own
// wavefront) plus the counts of the wavefronts before its own.  One block's chain of latencies bounds it.  Up to one chunk those
// counts are the histogram too, so that the ids are read once, with no atomics; with that and a ballot per bit of an id, where
// there was a round of exchange and ballot per distinct id, 1024 pairs of 32 experts take 8.2 -> 4.5 us (a launch alone is 2 to 3).
constexpr int kOrderThreads = 1024, kOrderWaves = kOrderThreads / 64;

// A lane's rank among the lanes before it with the same id (of `bits` bits), and each id's number of lanes into `count`: the lanes with the
// same id are those that agree in every bit, a ballot each.
__device__ __forceinline__ int wave_rank(bool live, uint32_t e, int bits, int lane, int32_t *count) {
    uint64_t same = __ballot(live);
    for (int b = 0; b < bits; b++) {
        const bool one = (e >> b & 1u) != 0;
        const uint64_t ones = __ballot(one);
        same &= one ? ones : ~ones;
    }
    const int rank = __popcll(same & ((1ull << lane) - 1ull));
    if (live && rank == 0) count[e] = __popcll(same);
    return rank;
}

// Places the pairs [chunk, chunk + 1024) of the block stably: `next[e]` is where expert e's next pair goes (advanced by
// the chunk's count); `wave_count` is scratch [wavefronts][experts].  A pair's rank among the equal ids before it in
// the chunk comes from wavefront ballots (lanes before it in its own wavefront) plus the counts of the wavefronts
// before its own.
__device__ __forceinline__ void place_chunk(const uint32_t *__restrict__ ids, int64_t pairs, int32_t experts, int64_t chunk,
                                            int32_t *next, int32_t *wave_count, uint32_t *__restrict__ order,
                                            uint32_t *__restrict__ restore, uint32_t *__restrict__ sorted_ids,
                                            uint32_t *__restrict__ tokens, uint32_t choices) {
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int64_t p = chunk + tid;
    const bool live = p < pairs;
    const uint32_t e = live ? min(ids[p], (uint32_t)(experts - 1)) : 0u;  // an id beyond the experts is clamped
    for (int i = tid; i < kOrderWaves * experts; i += kOrderThreads) wave_count[i] = 0;
    __syncthreads();
    const int rank = wave_rank(live, e, 32 - __clz(experts - 1), lane, wave_count + wave * experts);
    __syncthreads();
    if (live) {
        int before = 0;
        for (int w = 0; w < wave; w++) before += wave_count[w * experts + e];
        const uint32_t at = (uint32_t)(next[e] + before + rank);
        order[at] = (uint32_t)p;
        restore[p] = at;
        sorted_ids[at] = e;
        if (tokens != nullptr) tokens[at] = (uint32_t)p / choices;
    }
    __syncthreads();
    for (int ee = tid; ee < experts; ee += kOrderThreads) {
        int total = 0;
        for (int w = 0; w < kOrderWaves; w++) total += wave_count[w * experts + ee];
        next[ee] += total;
    }
    __syncthreads();
}

__global__ void __launch_bounds__(kOrderThreads)
moe_order_kernel(const uint32_t *__restrict__ ids, int64_t pairs, int32_t experts, uint32_t *__restrict__ order,
                 uint32_t *__restrict__ restore, uint32_t *__restrict__ sorted_ids, int32_t *__restrict__ offsets,
                 uint32_t *__restrict__ tokens, uint32_t choices) {
    extern __shared__ int32_t lds_i[];
    int32_t *next = lds_i;                       // [experts]: histogram, then where each expert's next pair goes
    int32_t *wave_count = lds_i + experts;       // [waves][experts]: this chunk's pairs per wavefront and expert
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    if (pairs <= kOrderThreads) {  // one chunk: its wavefronts' counts are the histogram
        const bool live = tid < pairs;
        const uint32_t e = live ? min(ids[tid], (uint32_t)(experts - 1)) : 0u;
        for (int i = tid; i < kOrderWaves * experts; i += kOrderThreads) wave_count[i] = 0;
        __syncthreads();
        const int rank = wave_rank(live, e, 32 - __clz(experts - 1), lane, wave_count + wave * experts);
        __syncthreads();
        if (wave == 0) {
            int32_t carry = 0;
            for (int base = 0; base < experts; base += 64) {
                const int ee = base + lane;
                int32_t c[kOrderWaves], count = 0;
#pragma unroll
                for (int w = 0; w < kOrderWaves; w++) c[w] = ee < experts ? wave_count[w * experts + ee] : 0;
#pragma unroll
                for (int w = 0; w < kOrderWaves; w++) {
                    const int32_t before = count;
                    count += c[w], c[w] = before;
                }
                int32_t incl = count;
#pragma unroll
                for (int d = 1; d < 64; d <<= 1) {
                    const int32_t up = __shfl_up(incl, d);
                    if (lane >= d) incl += up;
                }
                const int32_t first = carry + incl - count;
                if (ee < experts) {
                    offsets[ee] = first;
#pragma unroll
                    for (int w = 0; w < kOrderWaves; w++) wave_count[w * experts + ee] = first + c[w];
                }
                carry += __shfl(incl, 63);
            }
        }
        __syncthreads();
        if (live) {
            const uint32_t at = (uint32_t)(wave_count[wave * experts + e] + rank);
            order[at] = (uint32_t)tid;
            restore[tid] = at;
            sorted_ids[at] = e;
            if (tokens != nullptr) tokens[at] = (uint32_t)tid / choices;
        }
        return;
    }
    for (int e = tid; e < experts; e += kOrderThreads) next[e] = 0;
    __syncthreads();
    for (int64_t p = tid; p < pairs; p += kOrderThreads) atomicAdd(&next[min(ids[p], (uint32_t)(experts - 1))], 1);
    __syncthreads();
    // Exclusive scan by one wavefront, 64 experts at a time.
    if (wave == 0) {
        int32_t carry = 0;
        for (int base = 0; base < experts; base += 64) {
            const int e = base + lane;
            const int32_t count = e < experts ? next[e] : 0;
            int32_t incl = count;
#pragma unroll
            for (int d = 1; d < 64; d <<= 1) {
                const int32_t up = __shfl_up(incl, d);
                if (lane >= d) incl += up;
            }
            if (e < experts) {
                next[e] = carry + incl - count;
                offsets[e] = carry + incl - count;
            }
            carry += __shfl(incl, 63);
        }
    }
    __syncthreads();
    for (int64_t chunk = 0; chunk < pairs; chunk += kOrderThreads) place_chunk(ids, pairs, experts, chunk, next, wave_count, order, restore, sorted_ids, tokens, choices);
}

// The same ordering for many pairs, over the whole chip in three steps: every block counts the ids of its chunk of
// 1024 pairs; one block turns the counts into the experts' offsets and, per chunk and expert, the position of the
// chunk's first such pair (chunks in order: the sort stays stable); every block places its chunk.
__global__ void __launch_bounds__(kOrderThreads)
moe_count_kernel(const uint32_t *__restrict__ ids, int64_t pairs, int32_t experts, int32_t *__restrict__ counts) {
    extern __shared__ int32_t lds_i[];
    const int tid = threadIdx.x;
    for (int e = tid; e < experts; e += kOrderThreads) lds_i[e] = 0;
    __syncthreads();
    const int64_t p = (int64_t)blockIdx.x * kOrderThreads + tid;
    if (p < pairs) atomicAdd(&lds_i[min(ids[p], (uint32_t)(experts - 1))], 1);
    __syncthreads();
    for (int e = tid; e < experts; e += kOrderThreads) counts[(int64_t)blockIdx.x * experts + e] = lds_i[e];
}

__global__ void __launch_bounds__(kOrderThreads)
moe_scan_kernel(int32_t *__restrict__ counts, int32_t chunks, int32_t experts, int32_t *__restrict__ offsets) {
    extern __shared__ int32_t lds_i[];  // [experts]: totals, then offsets
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    for (int e = tid; e < experts; e += kOrderThreads) {
        int32_t total = 0;
        for (int c = 0; c < chunks; c++) total += counts[(int64_t)c * experts + e];
        lds_i[e] = total;
    }
    __syncthreads();
    if (wave == 0) {  // exclusive scan over the experts, 64 at a time
        int32_t carry = 0;
        for (int base = 0; base < experts; base += 64) {
            const int e = base + lane;
            const int32_t count = e < experts ? lds_i[e] : 0;
            int32_t incl = count;
#pragma unroll
            for (int d = 1; d < 64; d <<= 1) {
                const int32_t up = __shfl_up(incl, d);
                if (lane >= d) incl += up;
            }
            if (e < experts) {
                lds_i[e] = carry + incl - count;
                offsets[e] = carry + incl - count;
            }
            carry += __shfl(incl, 63);
        }
    }
    __syncthreads();
    for (int e = tid; e < experts; e += kOrderThreads) {
        int32_t at = lds_i[e];
        for (int c = 0; c < chunks; c++) {
            const int32_t n = counts[(int64_t)c * experts + e];
            counts[(int64_t)c * experts + e] = at;
            at += n;
        }
    }
}

__global__ void __launch_bounds__(kOrderThreads)
moe_place_kernel(const uint32_t *__restrict__ ids, int64_t pairs, int32_t experts, const int32_t *__restrict__ starts,
                 uint32_t *__restrict__ order, uint32_t *__restrict__ restore, uint32_t *__restrict__ sorted_ids,
                 uint32_t *__restrict__ tokens, uint32_t choices) {
    extern __shared__ int32_t lds_i[];
    int32_t *next = lds_i, *wave_count = lds_i + experts;
    for (int e = threadIdx.x; e < experts; e += kOrderThreads) next[e] = starts[(int64_t)blockIdx.x * experts + e];
    __syncthreads();
    place_chunk(ids, pairs, experts, (int64_t)blockIdx.x * kOrderThreads, next, wave_count, order, restore, sorted_ids, tokens, choices);
}

// round(a / b) in the element type.  The float32 quotient is correctly rounded and float32 carries more than twice
// the element types' digits, so rounding it again gives the correctly rounded quotient of the element type.
template <typename T> __device__ __forceinline__ float elem_div(float a, float b) {
    if constexpr (sizeof(T) == 4) return a / b;
    else if constexpr (Elem<T>::code == 10) return bf16_bits_to_f32(f32_to_bf16_bits(a / b));
    else return (float)(f16_t)(a / b);
}

// The order of the reference's sort: NaN last for float32 and half; bfloat16 compares plainly, as its sort does
// (crates/nuvec-kernels/src/metal/moe.metal:19-31).
template <typename T> __device__ __forceinline__ bool route_less(float a, float b) {
    if constexpr (Elem<T>::code != 10) {
        const bool an = a != a, bn = b != b;
        if (an | bn) return (!an) & bn;
    }
    return a < b;
}

// fast::moe_route (crates/nuvec-kernels/src/metal/moe.metal:33-88): of one row's `n` probabilities `p` the k largest in
// the stable ascending order, their values and, with `normalize`, those divided by their sum (summed in the
// element type, in order).  All threads of the block; an expert's position in the sorted row is the number of experts
// sorting before it.
template <typename T>
__device__ __forceinline__ void route_row(const float *p, float *top, float *total, uint32_t *__restrict__ indices, T *__restrict__ scores,
                                          int n, int k, int normalize) {
    for (int e = threadIdx.x; e < n; e += blockDim.x) {
        const float v = p[e];
        int rank = 0;
#pragma unroll 8
        for (int j = 0; j < n; j++) {
            const float u = p[j];
            rank += (route_less<T>(u, v) || (!route_less<T>(v, u) && j < e)) ? 1 : 0;
        }
        const int slot = rank - (n - k);
        if (slot >= 0) {
            indices[slot] = (uint32_t)e;
            top[slot] = v;
        }
    }
    __syncthreads();
    if (normalize) {
        if (threadIdx.x == 0) {
            float sum = 0.0f;
            for (int j = 0; j < k; j++) sum = Elem<T>::add(top[j], sum);
            *total = sum;
        }
        __syncthreads();
    }
    for (int e = threadIdx.x; e < k; e += blockDim.x) Elem<T>::store(scores, e, normalize ? elem_div<T>(top[e], *total) : top[e]);
}

// The same for up to 64 experts, every wavefront holding all of them, lane e expert e's `v`: a wavefront ranks every so manieth expert by
// two ballots (one wavefront and a comparison a turn: 1 us of a token's router; a thread an expert, with the probabilities read from
// LDS, as much).
template <typename T>
__device__ __forceinline__ void route_lanes(float v, float *top, uint32_t *__restrict__ indices, T *__restrict__ scores, int n, int k, int normalize) {
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), waves = blockDim.x >> 6;
    for (int e = wave; e < n; e += waves) {
        const float u = from_lane(v, e);
        const bool before = route_less<T>(v, u), level = !before && !route_less<T>(u, v);
        const int slot = __popcll(__ballot(before && lane < n)) + __popcll(__ballot(level && lane < e)) - (n - k);
        if (slot >= 0 && lane == 0) top[slot] = u, indices[slot] = (uint32_t)e;
    }
    __syncthreads();
    const int tid = threadIdx.x;
    if (tid >= k) return;
    float total = 0.0f;
    if (normalize)
        for (int j = 0; j < k; j++) total = Elem<T>::add(top[j], total);
    Elem<T>::store(scores, tid, normalize ? elem_div<T>(top[tid], total) : top[tid]);
}

// One block per row, one thread per expert.
template <typename T>
__global__ void __launch_bounds__(1024) moe_route_kernel(const T *__restrict__ probs, uint32_t *__restrict__ indices,
                                                         T *__restrict__ scores, int n, int k, int normalize) {
    __shared__ float p[1024], top[1024], total;
    const int64_t row = blockIdx.x;
    for (int e = threadIdx.x; e < n; e += blockDim.x) p[e] = Elem<T>::load(probs + row * n, e);
    __syncthreads();
    route_row<T>(p, top, &total, indices + row * k, scores + row * k, n, k, normalize);
}

// The router of a mixture-of-experts block in one launch (MoeMlp, crates/nuvec-lm/src/model.rs:2218-2272): logits of a token
// (float32 sums, rounded to the element type), their softmax (float32, rounded once), `moe_route`; and what the gathered
// products read beside its choices, the token of each pair and the pair's own number.  One block per token, a wavefront per
// two experts in turn: latency is the bound, of the 184 KB of a token's 32 x 2880 gate into one compute unit and of what follows, which up
// to 64 experts every wavefront does by itself (6.8 -> 5.7 us, gates from memory).  The library's product, two conversions, softmax and
// `moe_route` took 17.6 us of kernels at one token and 36 us at 256.
template <typename T>
__global__ void __launch_bounds__(1024) moe_router_kernel(const T *__restrict__ x, const T *__restrict__ gate, int dims, int n, int k, int normalize,
                                                          uint32_t *__restrict__ indices, T *__restrict__ scores,
                                                          uint32_t *__restrict__ tokens, uint32_t *__restrict__ identity) {
    constexpr int V = 16 / sizeof(T);  // values of a 16-byte load
    __shared__ float p[1024], top[1024], total;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, waves = blockDim.x >> 6;
    const int64_t row = blockIdx.x;
    const T *xr = x + row * dims;
    // Two experts a wavefront at a time and kChunks pieces of their rows and of x requested together: one token waits for little
    // else (one expert and up to four pieces at a time: 8.8 us for 32 experts of 2880 values).
    constexpr int kChunks = 6;
    for (int e = wave; e < n; e += 2 * waves) {
        const int e1 = e + waves < n ? e + waves : e;
        const T *g[2] = {gate + (int64_t)e * dims, gate + (int64_t)e1 * dims};
        float sum[2] = {0.0f, 0.0f};
        for (int c0 = lane * V; c0 < dims; c0 += kChunks * 64 * V) {
            uint4 xq[kChunks], gq[kChunks][2];
#pragma unroll
            for (int j = 0; j < kChunks; j++) {
                const int c = c0 + j * 64 * V < dims ? c0 + j * 64 * V : c0;  // (past the row: read again, not used)
                xq[j] = *reinterpret_cast<const uint4 *>(xr + c);
                gq[j][0] = *reinterpret_cast<const uint4 *>(g[0] + c), gq[j][1] = *reinterpret_cast<const uint4 *>(g[1] + c);
            }
#pragma unroll
            for (int j = 0; j < kChunks; j++) {
                if (c0 + j * 64 * V >= dims) continue;
                T xv[V], gv[2][V];
                __builtin_memcpy(xv, &xq[j], 16), __builtin_memcpy(gv[0], &gq[j][0], 16), __builtin_memcpy(gv[1], &gq[j][1], 16);
#pragma unroll
                for (int u = 0; u < 2; u++)
#pragma unroll
                    for (int i = 0; i < V; i++) sum[u] = __builtin_fmaf(Elem<T>::load(xv, i), Elem<T>::load(gv[u], i), sum[u]);
            }
        }
        sum[0] = wave_sum_lane63(sum[0]), sum[1] = wave_sum_lane63(sum[1]);
        if (lane == 63) p[e] = Elem<T>::mul(sum[0], 1.0f), p[e1] = Elem<T>::mul(sum[e1 == e ? 0 : 1], 1.0f);
    }
    __syncthreads();
    if (n <= 64) {
        const float logit = lane < n ? p[lane] : -INFINITY;
        const float power = expf(logit - from_lane(wave_max_lane63(logit), 63));
        const float share = Elem<T>::mul(power / from_lane(wave_sum_lane63(lane < n ? power : 0.0f), 63), 1.0f);
        if (tid < k) tokens[row * k + tid] = (uint32_t)row, identity[row * k + tid] = (uint32_t)(row * k + tid);
        route_lanes<T>(share, top, indices + row * k, scores + row * k, n, k, normalize);
        return;
    }
    if (wave == 0) {
        float most = -INFINITY, sum = 0.0f;
        for (int e = lane; e < n; e += 64) most = fmaxf(most, p[e]);
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) most = fmaxf(most, __shfl_xor(most, o));
        for (int e = lane; e < n; e += 64) sum += expf(p[e] - most);
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) sum += __shfl_xor(sum, o);
        for (int e = lane; e < n; e += 64) p[e] = Elem<T>::mul(expf(p[e] - most) / sum, 1.0f);
    }
    for (int j = tid; j < k; j += blockDim.x) tokens[row * k + j] = (uint32_t)row, identity[row * k + j] = (uint32_t)(row * k + j);
    __syncthreads();
    route_row<T>(p, top, &total, indices + row * k, scores + row * k, n, k, normalize);
}

// fast::weighted_sum (moe.metal:90-118): out[r, c] = sum over j of x[r, j, c] * w[r, j], every product and every
// addition rounded to the element type: min(k, 8) partial sums of every min(k, 8)-th product (one partial sum when
// D = 1), added in order.  One thread per V consecutive elements of a row (V = 1: rows that are not whole runs of V).
template <typename T, int V>
__global__ void __launch_bounds__(256) weighted_sum_kernel(const T *__restrict__ x, const T *__restrict__ w, T *__restrict__ out,
                                                           int64_t rows, int k, int64_t d) {
    struct __align__(V * sizeof(T)) Run { T v[V]; };
    const int64_t at = ((int64_t)blockIdx.x * 256 + threadIdx.x) * V;
    if (at >= rows * d) return;
    const int64_t r = at / d, c = at - r * d;
    x += r * k * d + c;
    w += r * k;
    auto load = [&](int j) { return *reinterpret_cast<const Run *>(x + (int64_t)j * d); };
    float sum[V];
    if (k <= 8 && d != 1) {  // a partial sum is one product: all rows requested at once
        Run run[8];
        float wj[8];
#pragma unroll
        for (int j = 0; j < 8; j++) run[j] = load(j < k ? j : k - 1), wj[j] = Elem<T>::load(w, j < k ? j : k - 1);
#pragma unroll
        for (int j = 0; j < 8; j++)
            if (j < k)
#pragma unroll
                for (int i = 0; i < V; i++) {
                    const float t = Elem<T>::add(Elem<T>::mul(Elem<T>::load(run[j].v, i), wj[j]), 0.0f);
                    sum[i] = j == 0 ? t : Elem<T>::add(t, sum[i]);
                }
    } else {
        const int lanes = d == 1 ? 1 : 8;
        for (int y = 0; y < lanes; y++) {
            float t[V];
#pragma unroll
            for (int i = 0; i < V; i++) t[i] = 0.0f;
            for (int j = y; j < k; j += lanes) {
                const Run run = load(j);
                const float wj = Elem<T>::load(w, j);
#pragma unroll
                for (int i = 0; i < V; i++) t[i] = Elem<T>::add(Elem<T>::mul(Elem<T>::load(run.v, i), wj), t[i]);
            }
#pragma unroll
            for (int i = 0; i < V; i++) sum[i] = y == 0 ? t[i] : Elem<T>::add(t[i], sum[i]);
        }
    }
    Run o;
#pragma unroll
    for (int i = 0; i < V; i++) Elem<T>::store(o.v, i, sum[i]);
    *reinterpret_cast<Run *>(out + at) = o;
}

__global__ void fill_zero_kernel(uint16_t *p, int64_t halves) {
    const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t < halves) p[t] = 0;
}

}  // namespace

int32_t launch_sorted_offsets(const uint32_t *indices, int64_t rows, int64_t m, int32_t groups, int32_t *offsets,
                              hipStream_t s) {
    const int64_t n = rows * groups;
    hipLaunchKernelGGL(sorted_offsets_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, indices, rows, m, groups, offsets);
    NVQ_LAUNCH_CHECK("sorted_offsets");
    return NVQ_OK;
}

size_t moe_order_lds_bytes(int32_t experts) { return (size_t)(1 + kOrderWaves) * experts * sizeof(int32_t); }

// Above this many pairs the ordering runs over the whole chip (three launches) when the caller gave the workspace.
constexpr int64_t kOrderOneBlock = 2048;
size_t moe_order_workspace_bytes(int64_t pairs, int32_t experts) {
    if (pairs <= kOrderOneBlock) return 0;
    return (size_t)((pairs + kOrderThreads - 1) / kOrderThreads) * (size_t)experts * sizeof(int32_t);
}

int32_t launch_moe_order(const uint32_t *ids, int64_t pairs, int32_t experts, uint32_t *order, uint32_t *restore,
                         uint32_t *sorted_ids, int32_t *offsets, uint32_t *tokens, int32_t choices, void *workspace, hipStream_t s) {
    if (workspace == nullptr || pairs <= kOrderOneBlock) {
        hipLaunchKernelGGL(moe_order_kernel, dim3(1), dim3(kOrderThreads), moe_order_lds_bytes(experts), s, ids, pairs, experts, order,
                           restore, sorted_ids, offsets, tokens, (uint32_t)choices);
        NVQ_LAUNCH_CHECK("moe_order");
        return NVQ_OK;
    }
    const unsigned chunks = (unsigned)((pairs + kOrderThreads - 1) / kOrderThreads);
    int32_t *counts = (int32_t *)workspace;
    hipLaunchKernelGGL(moe_count_kernel, dim3(chunks), dim3(kOrderThreads), (size_t)experts * sizeof(int32_t), s, ids, pairs, experts, counts);
    NVQ_LAUNCH_CHECK("moe_order (count)");
    hipLaunchKernelGGL(moe_scan_kernel, dim3(1), dim3(kOrderThreads), (size_t)experts * sizeof(int32_t), s, counts, (int32_t)chunks, experts, offsets);
    NVQ_LAUNCH_CHECK("moe_order (scan)");
    hipLaunchKernelGGL(moe_place_kernel, dim3(chunks), dim3(kOrderThreads), moe_order_lds_bytes(experts), s, ids, pairs, experts, counts, order,
                       restore, sorted_ids, tokens, (uint32_t)choices);
    NVQ_LAUNCH_CHECK("moe_order (place)");
    return NVQ_OK;
}

int32_t launch_moe_route(int32_t dtype, const void *probs, int64_t rows, int32_t experts, int32_t k, int32_t normalize,
                         uint32_t *indices, void *scores, hipStream_t s) {
    const dim3 grid((unsigned)rows), block((unsigned)((experts + 63) / 64 * 64));
    if (dtype == NVQ_F32)
        hipLaunchKernelGGL(moe_route_kernel<float>, grid, block, 0, s, (const float *)probs, indices, (float *)scores, experts, k, normalize);
    else if (dtype == NVQ_BF16)
        hipLaunchKernelGGL(moe_route_kernel<bf16_t>, grid, block, 0, s, (const bf16_t *)probs, indices, (bf16_t *)scores, experts, k, normalize);
    else
        hipLaunchKernelGGL(moe_route_kernel<f16_t>, grid, block, 0, s, (const f16_t *)probs, indices, (f16_t *)scores, experts, k, normalize);
    NVQ_LAUNCH_CHECK("moe_route");
    return NVQ_OK;
}

template <typename T>
static void run_weighted_sum(const void *x, const void *w, int64_t rows, int32_t k, int64_t d, void *out, hipStream_t s) {
    // runs of 8 bytes where the rows are whole runs of them and every operand is aligned to one
    constexpr int V = 8 / (int)sizeof(T);
    const bool runs = d % V == 0 && (((uintptr_t)x | (uintptr_t)out) & 7) == 0;
    const dim3 grid((unsigned)((rows * d / (runs ? V : 1) + 255) / 256)), block(256);
    if (runs) hipLaunchKernelGGL((weighted_sum_kernel<T, V>), grid, block, 0, s, (const T *)x, (const T *)w, (T *)out, rows, k, d);
    else hipLaunchKernelGGL((weighted_sum_kernel<T, 1>), grid, block, 0, s, (const T *)x, (const T *)w, (T *)out, rows, k, d);
}

int32_t launch_weighted_sum(int32_t dtype, const void *x, const void *w, int64_t rows, int32_t k, int64_t d, void *out, hipStream_t s) {
    if (dtype == NVQ_F32) run_weighted_sum<float>(x, w, rows, k, d, out, s);
    else if (dtype == NVQ_BF16) run_weighted_sum<bf16_t>(x, w, rows, k, d, out, s);
    else run_weighted_sum<f16_t>(x, w, rows, k, d, out, s);
    NVQ_LAUNCH_CHECK("weighted_sum");
    return NVQ_OK;
}

template <typename T>
static void run_moe_router(const void *x, const void *gate, int64_t rows, int32_t dims, int32_t experts, int32_t k, int32_t normalize,
                           uint32_t *indices, void *scores, uint32_t *tokens, uint32_t *identity, hipStream_t s) {
    const int waves = experts < 16 ? (experts < 4 ? 4 : experts) : 16;
    hipLaunchKernelGGL(moe_router_kernel<T>, dim3((unsigned)rows), dim3(64 * waves), 0, s, (const T *)x, (const T *)gate, dims, experts, k, normalize,
                       indices, (T *)scores, tokens, identity);
}

int32_t launch_moe_router(int32_t dtype, const void *x, const void *gate, int64_t rows, int32_t dims, int32_t experts, int32_t k,
                          int32_t normalize, uint32_t *indices, void *scores, uint32_t *tokens, uint32_t *identity, hipStream_t s) {
    if (dtype == NVQ_F32) run_moe_router<float>(x, gate, rows, dims, experts, k, normalize, indices, scores, tokens, identity, s);
    else if (dtype == NVQ_BF16) run_moe_router<bf16_t>(x, gate, rows, dims, experts, k, normalize, indices, scores, tokens, identity, s);
    else run_moe_router<f16_t>(x, gate, rows, dims, experts, k, normalize, indices, scores, tokens, identity, s);
    NVQ_LAUNCH_CHECK("moe_router");
    return NVQ_OK;
}

// Zero-fills `bytes` (even: element sizes are 2 or 4) with a kernel, so that a caller capturing
// the stream into a graph records no memset node.
int32_t launch_fill_zero(void *p, int64_t bytes, hipStream_t s) {
    const int64_t halves = bytes / 2;
    hipLaunchKernelGGL(fill_zero_kernel, dim3((unsigned)((halves + 255) / 256)), dim3(256), 0, s, (uint16_t *)p, halves);
    NVQ_LAUNCH_CHECK("fill_zero");
    return NVQ_OK;
}

}  // namespace nvq
