// The gated activation between the experts' up / gate products and their down product, in one pass over the two
// products: each row's expert's bias added to either (the reference's `SwitchProjection::forward`,
// crates/nuvec-lm/src/model.rs:2139-2143: `y + bias[indices]`), then SwiGLU or gpt-oss's clamped SwiGLU
// (`SwitchGlu::through`, model.rs:2157-2170; crates/nuvec-nn/src/lib.rs:513-519 `silu(gate) * x` with
// `silu(x) = x * sigmoid(x)` lib.rs:343-345, and lib.rs:564-570).  The reference evaluates the graph one operation
// at a time, each result an array of the activations' type (crates/nuvec-core/src/fused.rs:190-215), so every
// operation below rounds to that type; sigmoid is kernels.rs:1539-1543 in float32.
#include "nvq_device.h"
#include "nvq_internal.h"

namespace nvq {
namespace {

// V consecutive outputs of a row a thread: one, or 16 bytes of each operand.  Bound by memory for many rows, which one output a thread,
// a 64-bit division for its row included, left to half (us, bfloat16: 2048 rows of 14336 80 -> 44, 517 rows of 4096 6.4 -> 5.2), by a
// launch's latency for few, which eight outputs one after the other make longer (64 rows of 4096 2.75 -> 3.06, kept at one).
template <typename T, int ACT, int V>
__global__ void __launch_bounds__(256) glu_kernel(const T *__restrict__ gate, const T *__restrict__ up, const T *__restrict__ gate_bias,
                                                  const T *__restrict__ up_bias, const int32_t *__restrict__ ids, T *__restrict__ out,
                                                  int64_t rows, int64_t hidden, int64_t gate_stride, int64_t up_stride, int64_t experts,
                                                  float alpha, float limit) {
    struct __align__(V * sizeof(T)) Run { T v[V]; };
    const int64_t idx = ((int64_t)blockIdx.x * 256 + threadIdx.x) * V;
    if (idx >= rows * hidden) return;
    const int64_t r = idx / hidden, c = idx - r * hidden;
    auto run = [](const T *p) { return *reinterpret_cast<const Run *>(p); };
    const Run gate_run = run(gate + r * gate_stride + c), up_run = run(up + r * up_stride + c);
    Run gate_add, up_add, result;
    if (gate_bias != nullptr) {
        int64_t e = ids[r];  // an id outside the biases is the caller's error: clamped
        e = e < 0 ? 0 : (e >= experts ? experts - 1 : e);
        gate_add = run(gate_bias + e * hidden + c), up_add = run(up_bias + e * hidden + c);
    }
#pragma unroll
    for (int i = 0; i < V; i++) {
        float g = Elem<T>::load(gate_run.v, i), u = Elem<T>::load(up_run.v, i);
        if (gate_bias != nullptr) g = Elem<T>::add(g, Elem<T>::load(gate_add.v, i)), u = Elem<T>::add(u, Elem<T>::load(up_add.v, i));
        Elem<T>::store(result.v, i, glu<T, ACT>(g, u, alpha, limit));
    }
    *reinterpret_cast<Run *>(out + idx) = result;
}

template <typename T, int V>
int32_t run_glu_runs(const nvq_glu_desc &d, const void *gate, const void *up, const void *gate_bias, const void *up_bias, const int32_t *ids,
                     void *out, hipStream_t s) {
    const dim3 grid((unsigned)((d.rows * d.hidden + 256 * V - 1) / (256 * V)));
    void (*kernel)(const T *, const T *, const T *, const T *, const int32_t *, T *, int64_t, int64_t, int64_t, int64_t, int64_t, float, float) =
        d.activation == NVQ_GLU_SWIGLU       ? glu_kernel<T, NVQ_GLU_SWIGLU, V>
        : d.activation == NVQ_GLU_SWIGLU_OAI ? glu_kernel<T, NVQ_GLU_SWIGLU_OAI, V>
                                             : glu_kernel<T, NVQ_GLU_GEGLU, V>;
    hipLaunchKernelGGL(kernel, grid, dim3(256), 0, s, (const T *)gate, (const T *)up, (const T *)gate_bias, (const T *)up_bias, ids, (T *)out, d.rows,
                       d.hidden, d.gate_stride, d.up_stride, d.experts, d.alpha, d.limit);
    NVQ_LAUNCH_CHECK("glu");
    return NVQ_OK;
}

template <typename T>
int32_t run_glu(const nvq_glu_desc &d, const void *gate, const void *up, const void *gate_bias, const void *up_bias, const int32_t *ids,
                void *out, hipStream_t s) {
    constexpr int V = 16 / sizeof(T);
    const uintptr_t pointers = (uintptr_t)gate | (uintptr_t)up | (uintptr_t)gate_bias | (uintptr_t)up_bias | (uintptr_t)out;
    const bool whole = d.rows * d.hidden >= 1 << 20 && pointers % 16 == 0 && d.hidden % V == 0 && d.gate_stride % V == 0 && d.up_stride % V == 0;
    return whole ? run_glu_runs<T, V>(d, gate, up, gate_bias, up_bias, ids, out, s) : run_glu_runs<T, 1>(d, gate, up, gate_bias, up_bias, ids, out, s);
}

}  // namespace

int32_t launch_glu(const nvq_glu_desc &d, const void *gate, const void *up, const void *gate_bias, const void *up_bias,
                   const int32_t *ids, void *out, hipStream_t s) {
    switch (d.dtype) {
    case NVQ_F32: return run_glu<float>(d, gate, up, gate_bias, up_bias, ids, out, s);
    case NVQ_BF16: return run_glu<bf16_t>(d, gate, up, gate_bias, up_bias, ids, out, s);
    default: return run_glu<f16_t>(d, gate, up, gate_bias, up_bias, ids, out, s);
    }
}

}  // namespace nvq
