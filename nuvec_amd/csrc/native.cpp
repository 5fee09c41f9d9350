// The Python package's calls in native code: `nuvec_amd._native`.
//
// A decode step is launch-bound: its kernels take 3 to 20 us each, and the argument checks, descriptors and allocations of
// one call took 12 to 17 us in Python (a one-row product of W[1024,4096]: 16.7 us per call, of which the kernel is 3.4).  Here
// the same work is done on the tensors' own C++ objects, a block's layers in one call.
//
// Every function takes the plain case alone: operands on the bound device, dense, of one element type, of matching shapes, and
// layers whose methods are the package's own.  Whatever else it meets (and whatever the library refuses) it declines by returning
// None, and the caller's Python path, which holds every conversion and the reference's messages, does the call.  The operands of
// every product of a block are looked at before the first is launched; where the library itself refuses a later one, what ran
// before it has written intermediate tensors that are dropped.
//
// The interpreter lock is released while a call allocates and launches, as ctypes and torch's own operators release it.
#include <torch/csrc/Dtype.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

#include <ATen/hip/EmptyTensor.h>
#include <ATen/core/Tensor.h>
#include <c10/hip/HIPFunctions.h>
#include <c10/hip/HIPStream.h>

#include <atomic>
#include <vector>

#include "nuvec_hip.h"

namespace {

using at::Tensor;

// ── reading Python objects ──────────────────────────────────────────────────────────────────────────────────────────
struct Names {
    PyObject *mode, *group_size, *bits, *weight, *scales, *biases, *bias, *quant, *global_scale;
    PyObject *gate_proj, *up_proj, *down_proj, *gate_up_proj, *geglu;
    PyObject *gate, *switch_mlp, *experts_per_token, *norm_topk_prob, *gate_up_paired, *activation, *alpha, *limit;
} names;

std::atomic<uint64_t> ready_devices{0};  // devices nvq_init has answered for (ops._init)

struct Ref {
    PyObject *p;
    explicit Ref(PyObject *o) : p(o) {}
    Ref(const Ref &) = delete;
    ~Ref() { Py_XDECREF(p); }
};

bool declined() {
    PyErr_Clear();
    return false;
}

// A class of `layers` and the methods of it that a call here stands in for.  An object is plain if it is of that very class
// (a subclass may have others), the class still holds the functions it was defined with, and the object has none of its own.
struct Kind {
    PyTypeObject *type = nullptr;
    std::vector<std::pair<PyObject *, PyObject *>> methods;  // name, function

    bool plain(PyObject *o) const {
        if (type == nullptr || Py_TYPE(o) != type) return false;
        PyObject **own = _PyObject_GetDictPtr(o);
        for (const auto &m : methods) {
            if (PyDict_GetItemWithError(type->tp_dict, m.first) != m.second) return declined();
            if (own != nullptr && *own != nullptr && PyDict_GetItemWithError(*own, m.first) != nullptr) return false;
        }
        return true;
    }
};
Kind linear_kind, projection_kind, switch_glu_kind, moe_kind;

bool read_int(PyObject *o, PyObject *name, int32_t &v) {
    Ref a(PyObject_GetAttr(o, name));
    if (a.p == nullptr || !PyLong_Check(a.p)) return declined();
    const long n = PyLong_AsLong(a.p);
    if (n == -1 && PyErr_Occurred()) return declined();
    v = (int32_t)n;
    return true;
}

bool read_quant(PyObject *o, nvq_quant &q) {
    return read_int(o, names.mode, q.mode) && read_int(o, names.group_size, q.group_size) && read_int(o, names.bits, q.bits);
}

bool read_float(PyObject *o, PyObject *name, float &v) {
    Ref a(PyObject_GetAttr(o, name));
    if (a.p == nullptr) return declined();
    const double d = PyFloat_AsDouble(a.p);
    if (d == -1.0 && PyErr_Occurred()) return declined();
    v = (float)d;
    return true;
}

bool read_truth(PyObject *o, PyObject *name, bool &v) {
    Ref a(PyObject_GetAttr(o, name));
    const int t = a.p == nullptr ? -1 : PyObject_IsTrue(a.p);
    if (t < 0) return declined();
    v = t != 0;
    return true;
}

// A tensor, or none at all for None.
bool as_tensor(PyObject *o, Tensor &t) {
    if (o == Py_None) return true;
    if (!THPVariable_Check(o)) return false;
    t = THPVariable_Unpack(o);
    return true;
}
bool read_tensor(PyObject *o, PyObject *name, Tensor &t) {
    Ref a(PyObject_GetAttr(o, name));
    return a.p == nullptr ? declined() : as_tensor(a.p, t);
}

// ── operands ────────────────────────────────────────────────────────────────────────────────────────────────────────
int32_t code_of(at::ScalarType t) {
    switch (t) {
    case at::kHalf: return NVQ_F16;
    case at::kBFloat16: return NVQ_BF16;
    case at::kFloat: return NVQ_F32;
    default: return -1;
    }
}

bool is_word(at::ScalarType t) { return t == at::kUInt32 || t == at::kInt; }

const void *ptr(const Tensor &t) { return t.defined() ? t.const_data_ptr() : nullptr; }

// Whether `t` lies densely on the device that the library is bound to and that is current.
struct Place {
    c10::Device device;
    explicit Place(const Tensor &x) : device(x.defined() ? x.device() : c10::Device(at::kCPU)) {}
    bool usable() const {
        return device.is_cuda() && device.index() >= 0 && device.index() < 64 && (ready_devices >> device.index() & 1) != 0 &&
               c10::hip::current_device() == device.index();
    }
    bool holds(const Tensor &t) const { return t.device() == device && t.is_contiguous(); }
    void *stream() const { return c10::hip::getCurrentHIPStream(device.index()).stream(); }
    Tensor empty(at::IntArrayRef sizes, at::ScalarType type) const {
        return at::detail::empty_cuda(sizes, type, device, std::nullopt);
    }
};

struct Packed {
    Tensor w, s, b;
    nvq_quant q;

    // Codes, scales and biases of `dims` dimensions that go together and with activations of `type` (ops._check_groups,
    // ops._quantized_columns); `columns`: the values of a packed row.
    bool fits(const Place &at, at::ScalarType type, int64_t dims, int64_t &columns) const {
        if (!w.defined() || !s.defined() || !is_word(w.scalar_type()) || w.dim() != dims || s.dim() != dims || !at.holds(w) || !at.holds(s))
            return false;
        if (q.mode == NVQ_AFFINE) {
            if (!b.defined() || s.scalar_type() != type || b.scalar_type() != type || !at.holds(b) || b.sizes() != s.sizes()) return false;
        } else if (b.defined() || s.scalar_type() != at::kByte) {
            return false;
        }
        for (int64_t i = 0; i + 1 < dims; i++)
            if (w.size(i) != s.size(i)) return false;
        columns = s.size(dims - 1) * q.group_size;
        return columns > 0 && w.size(dims - 1) * 32 == columns * q.bits;
    }
};

bool bias_fits(const Tensor &bias, const Place &at, at::ScalarType type, int64_t n) {
    return !bias.defined() || (bias.scalar_type() == type && bias.dim() == 1 && bias.size(0) == n && at.holds(bias));
}

using Sizes = c10::SmallVector<int64_t, 6>;
Sizes with_last(at::IntArrayRef sizes, int64_t last) {
    Sizes s(sizes.begin(), sizes.end());
    s.back() = last;
    return s;
}

// ── the calls ───────────────────────────────────────────────────────────────────────────────────────────────────────
struct Flags {
    bool transpose = true, row_exact = false, rows = false, scratch = true;
};

// ops.quantized_matmul of one weight matrix.
bool product(const Tensor &x, const Packed &p, const Tensor &bias, Flags f, Tensor &out) {
    const Place at(x);
    if (!at.usable() || x.dim() < 2 || !x.is_contiguous() || x.numel() == 0) return false;
    const int32_t code = code_of(x.scalar_type());
    int64_t columns;
    if (code < 0 || !p.fits(at, x.scalar_type(), 2, columns)) return false;
    const int64_t rows = p.w.size(0), inner = f.transpose ? columns : rows, outer = f.transpose ? rows : columns;
    if (x.size(-1) != inner || outer == 0 || !bias_fits(bias, at, x.scalar_type(), outer)) return false;
    nvq_qmm_desc d{};
    d.quant = p.q, d.dtype = code, d.transpose = f.transpose, d.row_exact = f.row_exact, d.rows = f.rows;
    d.m = x.numel() / inner, d.n = outer, d.k = inner, d.item_rows = x.size(-2);
    const size_t need = f.scratch ? nvq_quantized_matmul_workspace_bytes(&d) : 0;
    Tensor workspace, y = at.empty(with_last(x.sizes(), outer), x.scalar_type());
    if (need > 0) workspace = at.empty({(int64_t)need}, at::kByte);
    const int32_t rc = nvq_quantized_linear(&d, ptr(x), ptr(p.w), ptr(p.s), ptr(p.b), ptr(bias), y.mutable_data_ptr(),
                                            need > 0 ? workspace.mutable_data_ptr() : nullptr, at.stream());
    if (rc != NVQ_OK) return false;
    out = std::move(y);
    return true;
}

nvq_qmm_desc gated_desc(const Tensor &x, int32_t code, const nvq_quant &q, int64_t n) {
    nvq_qmm_desc d{};
    d.quant = q, d.dtype = code, d.transpose = 1;
    d.m = x.numel() / x.size(-1), d.n = n, d.k = x.size(-1), d.item_rows = x.dim() > 1 ? x.size(-2) : 1;
    return d;
}

// The kernel of several gated rows that nvq_quantized_matmul_glu_several_takes names, and its workspace.
struct Several {
    int32_t kernel = 0;
    size_t need = 0;
};

// ops.quantized_matmul_glu, or (`several`) ops.quantized_matmul_glu_grouped or ops.quantized_matmul_glu_rows.  `asked`: what the
// question gave for a pair of these sizes, which costs as much as a launch.
bool product_glu(const Tensor &x, const Packed &p, const Tensor &bias, int32_t activation, float alpha, float limit, bool several,
                 const Several *asked, Tensor &out) {
    const Place at(x);
    if (!at.usable() || x.dim() < 1 || !x.is_contiguous() || x.numel() == 0) return false;
    const int32_t code = code_of(x.scalar_type());
    int64_t columns;
    if (code < 0 || !p.fits(at, x.scalar_type(), 2, columns) || x.size(-1) != columns) return false;
    const int64_t n = p.w.size(0);
    if (n == 0 || n % 128 != 0 || !bias_fits(bias, at, x.scalar_type(), n)) return false;
    const nvq_qmm_desc d = gated_desc(x, code, p.q, n);
    Several to;
    if (several && asked != nullptr) to = *asked;
    else if (several) to.kernel = nvq_quantized_matmul_glu_several_takes(&d, &to.need);
    if (several && to.kernel == 0) return false;
    const bool grouped = to.kernel == 1;
    const size_t need = to.need;
    Tensor workspace, y = at.empty(with_last(x.sizes(), n / 2), x.scalar_type());
    if (need > 0) workspace = at.empty({(int64_t)need}, at::kByte);
    const int32_t rc = grouped   ? nvq_quantized_matmul_glu_grouped(&d, activation, alpha, limit, ptr(x), ptr(p.w), ptr(p.s), ptr(p.b), ptr(bias),
                                                                    y.mutable_data_ptr(), at.stream())
                       : several ? nvq_quantized_matmul_glu_rows(&d, activation, alpha, limit, ptr(x), ptr(p.w), ptr(p.s), ptr(p.b), ptr(bias),
                                                               y.mutable_data_ptr(), need > 0 ? workspace.mutable_data_ptr() : nullptr, at.stream())
                               : nvq_quantized_matmul_glu(&d, activation, alpha, limit, ptr(x), ptr(p.w), ptr(p.s), ptr(p.b), ptr(bias),
                                                          y.mutable_data_ptr(), at.stream());
    if (rc != NVQ_OK) return false;
    out = std::move(y);
    return true;
}

struct Activation {
    int32_t code = NVQ_GLU_SWIGLU;
    float alpha = 0.0f, limit = 0.0f;
};

// ops.glu of two dense tensors, without biases.
bool gated(const Tensor &gate, const Tensor &up, int32_t activation, Tensor &out) {
    const Place at(gate);
    const int64_t hidden = gate.size(-1);
    nvq_glu_desc d{code_of(gate.scalar_type()), activation, 0.0f, 0.0f, gate.numel() / hidden, hidden, hidden, hidden, 0};
    Tensor y = at.empty(gate.sizes(), gate.scalar_type());
    if (nvq_glu(&d, ptr(gate), ptr(up), nullptr, nullptr, nullptr, y.mutable_data_ptr(), at.stream()) != NVQ_OK) return false;
    out = std::move(y);
    return true;
}

// ── mixture of experts ──────────────────────────────────────────────────────────────────────────────────────────────
struct Projection {  // layers.SwitchProjection: a packed weight and perhaps a bias per expert
    Packed p;
    Tensor bias;
    int64_t columns = 0, rows = 0;

    bool fits(const Place &at, at::ScalarType type, int64_t experts) {
        if (!p.fits(at, type, 3, columns) || p.w.size(0) != experts) return false;
        rows = p.w.size(1);
        return rows > 0 && (!bias.defined() || (bias.scalar_type() == type && bias.dim() == 2 && bias.size(0) == experts &&
                                                bias.size(1) == rows && at.holds(bias)));
    }
};

// The pairs of a pass: which row of x and which expert each takes, in the order they run.
struct Pairs {
    int64_t count, experts;
    const uint32_t *expert;       // of each pair, in order
    const int32_t *offsets;       // sorted by expert: where each expert's pairs start; NULL: any order
};

// One projection of all pairs (ops.gather_qmm, ops.gather_qmm_grouped): pair z takes row `from[z]` of x [x_rows, columns] and
// writes row `to[z]` (NULL: z).
bool project(const Place &at, const Tensor &x, int64_t x_rows, const Projection &w, const Pairs &pairs, const uint32_t *from, const uint32_t *to,
             bool with_bias, Tensor &out) {
    const nvq_gather_desc d{w.p.q, code_of(x.scalar_type()), 1, 0, 1, 1, w.rows, w.columns, pairs.count, x_rows, pairs.experts};
    Tensor y = at.empty({pairs.count, w.rows}, x.scalar_type());
    if (nvq_gather_qmm_expert_bias(&d, ptr(x), ptr(w.p.w), ptr(w.p.s), ptr(w.p.b), nullptr, from, pairs.expert, pairs.offsets, to,
                                   with_bias ? ptr(w.bias) : nullptr, y.mutable_data_ptr(), nullptr, at.stream()) != NVQ_OK)
        return false;
    out = std::move(y);
    return true;
}

struct Experts {  // layers.SwitchGlu
    Projection gate, up, down, both;
    bool fused = false, paired = false;
    Activation act;
};

// The pairs' gated hidden states (layers.SwitchGlu.forward up to the down projection).
bool hidden_states(const Place &at, const Tensor &x, int64_t x_rows, Experts &e, const Pairs &pairs, const uint32_t *tokens, Tensor &out) {
    const at::ScalarType type = x.scalar_type();
    const int64_t hidden = e.down.columns;
    if (e.fused && e.paired) {
        const nvq_gather_desc d{e.both.p.q, code_of(type), 1, 0, 1, 1, e.both.rows, e.both.columns, pairs.count, x_rows, pairs.experts};
        Tensor y = at.empty({pairs.count, hidden}, type);
        if (nvq_gather_qmm_glu(&d, e.act.code, e.act.alpha, e.act.limit, ptr(x), ptr(e.both.p.w), ptr(e.both.p.s), ptr(e.both.p.b), tokens,
                               pairs.expert, pairs.offsets, ptr(e.both.bias), y.mutable_data_ptr(), at.stream()) == NVQ_OK) {
            out = std::move(y);
            return true;
        }
    }
    // products without their biases, then biases and activation in one pass
    Tensor gate, up;
    int64_t stride = hidden;
    const char *second;
    if (e.fused && !e.paired) {
        if (!project(at, x, x_rows, e.both, pairs, tokens, nullptr, false, gate)) return false;
        stride = 2 * hidden;
        second = (const char *)ptr(gate) + hidden * gate.element_size();
    } else {
        if (!project(at, x, x_rows, e.gate, pairs, tokens, nullptr, false, gate) || !project(at, x, x_rows, e.up, pairs, tokens, nullptr, false, up))
            return false;
        second = (const char *)ptr(up);
    }
    const bool biased = e.gate.bias.defined();
    const nvq_glu_desc d{code_of(type), e.act.code, e.act.alpha, e.act.limit, pairs.count, hidden, stride, stride, biased ? pairs.experts : 0};
    Tensor y = at.empty({pairs.count, hidden}, type);
    if (nvq_glu(&d, ptr(gate), second, ptr(e.gate.bias), ptr(e.up.bias), biased ? (const int32_t *)pairs.expert : nullptr, y.mutable_data_ptr(),
                at.stream()) != NVQ_OK)
        return false;
    out = std::move(y);
    return true;
}

// layers.SwitchGlu._ordered.
bool pairs_ordered(const Experts &e, int32_t code, int64_t tokens, int64_t choices, int64_t experts) {
    if (tokens * choices >= 64) return true;
    const int64_t size = e.up.rows * e.up.columns;
    auto rule = [&](const Projection &w, int64_t values) { return nvq_moe_ordered(&w.p.q, code, tokens, (int32_t)choices, experts, values, 0) != 0; };
    if (!rule(e.up, 3 * size)) return false;
    const Projection *taken[3];
    int count = 0;
    for (const Projection *w : {&e.gate, &e.up, &e.down}) {
        const nvq_gather_desc d{w->p.q, code, 1, 0, 1, 1, w->rows, w->columns, tokens * choices, tokens * choices, experts};
        if (nvq_gather_sorted_takes(&d)) taken[count++] = w;
    }
    for (int i = 0; i < count; i++)
        if (!rule(*taken[i], count * size)) return false;
    return count > 0;
}

// layers.MoeMlp.forward.
bool moe(const Tensor &x, const Tensor &router, int64_t k, bool normalize, Experts &e, Tensor &out) {
    const Place at(x);
    if (!at.usable() || x.dim() != 3 || x.numel() == 0 || !x.is_contiguous()) return false;
    const at::ScalarType type = x.scalar_type();
    const int32_t code = code_of(type);
    if (code < 0 || !router.defined() || router.scalar_type() != type || router.dim() != 2 || !at.holds(router) || router.size(1) != x.size(2))
        return false;
    const int64_t rows = x.size(0) * x.size(1), dims = x.size(2), experts = router.size(0);
    if (k < 1 || k > experts || k >= 32 || dims > INT32_MAX || experts > 1024 || rows > INT32_MAX / k) return false;
    if (!e.gate.fits(at, type, experts) || !e.up.fits(at, type, experts) || !e.down.fits(at, type, experts)) return false;
    const int64_t hidden = e.down.columns;
    if (e.gate.columns != dims || e.up.columns != dims || e.gate.rows != hidden || e.up.rows != hidden ||
        e.gate.bias.defined() != e.up.bias.defined())
        return false;
    if (e.fused && (!e.both.fits(at, type, experts) || e.both.columns != dims || e.both.rows != 2 * hidden ||
                    e.both.bias.defined() != e.gate.bias.defined() || (e.paired && hidden % 64 != 0)))
        return false;

    const int64_t pairs = rows * k;
    void *stream = at.stream();
    // choices, tokens and numbers of the pairs; for ordered pairs the order, its inverse, sorted experts and tokens, the offsets
    const bool ordered = pairs_ordered(e, code, rows, k, experts);
    Tensor index = at.empty({pairs * (ordered ? 7 : 3) + (ordered ? experts : 0)}, at::kInt), scores = at.empty({rows, k}, type);
    uint32_t *chosen = (uint32_t *)index.mutable_data_ptr(), *tokens = chosen + pairs, *identity = tokens + pairs;
    if (nvq_moe_router(code, ptr(x), ptr(router), rows, (int32_t)dims, (int32_t)experts, (int32_t)k, normalize, chosen, scores.mutable_data_ptr(),
                       tokens, identity, stream) != NVQ_OK)
        return false;
    Pairs p{pairs, experts, chosen, nullptr};
    const uint32_t *to = nullptr;
    Tensor workspace, h, y;
    if (ordered) {
        uint32_t *order = identity + pairs, *restore = order + pairs, *sorted = restore + pairs, *sorted_tokens = sorted + pairs;
        int32_t *offsets = (int32_t *)(sorted_tokens + pairs);
        const size_t need = nvq_moe_order_workspace_bytes(pairs, (int32_t)experts);
        if (need > 0) workspace = at.empty({(int64_t)need}, at::kByte);
        if (nvq_moe_order_tokens(chosen, pairs, (int32_t)experts, (int32_t)k, order, restore, sorted, offsets, sorted_tokens,
                                 need > 0 ? workspace.mutable_data_ptr() : nullptr, stream) != NVQ_OK)
            return false;
        p.expert = sorted, p.offsets = offsets;
        tokens = sorted_tokens, to = order;
    }
    if (!hidden_states(at, x, rows, e, p, tokens, h) || e.down.rows == 0) return false;
    Tensor sum = at.empty({x.size(0), x.size(1), e.down.rows}, type);
    if (!ordered) {  // (few tokens: the down products with their sum)
        const nvq_gather_desc d{e.down.p.q, code, 1, 0, 0, 1, e.down.rows, hidden, pairs, pairs, experts};
        if (nvq_gather_qmm_sum_takes(&d, (int32_t)k) &&
            nvq_gather_qmm_sum(&d, ptr(h), ptr(e.down.p.w), ptr(e.down.p.s), ptr(e.down.p.b), nullptr, identity, chosen, ptr(e.down.bias), ptr(scores),
                               (int32_t)k, sum.mutable_data_ptr(), stream) == NVQ_OK) {
            out = std::move(sum);
            return true;
        }
    }
    if (!project(at, h, pairs, e.down, p, identity, to, true, y)) return false;
    if (nvq_weighted_sum(code, ptr(y), ptr(scores), rows, (int32_t)k, e.down.rows, sum.mutable_data_ptr(), stream) != NVQ_OK) return false;
    out = std::move(sum);
    return true;
}

// ── layers ──────────────────────────────────────────────────────────────────────────────────────────────────────────
struct Linear {
    Packed p;
    Tensor bias;
};
bool read_linear(PyObject *o, Linear &l) {
    if (!linear_kind.plain(o)) return false;
    if (!read_tensor(o, names.weight, l.p.w) || !read_tensor(o, names.scales, l.p.s) || !read_tensor(o, names.biases, l.p.b) ||
        !read_tensor(o, names.bias, l.bias))
        return false;
    Ref q(PyObject_GetAttr(o, names.quant));
    return q.p == nullptr ? declined() : read_quant(q.p, l.p.q);
}
bool read_linear(PyObject *o, PyObject *name, Linear &l) {
    Ref a(PyObject_GetAttr(o, name));
    return a.p == nullptr ? declined() : read_linear(a.p, l);
}

PyObject *none() { Py_RETURN_NONE; }

// A refusal inside torch (no memory left) is Python's exception, as it is where Python allocates.
template <typename F>
PyObject *guarded(F &&f) {
    try {
        return f();
    } catch (...) {  // (torch.OutOfMemoryError among them)
        torch::translate_exception_to_python(std::current_exception());
        return nullptr;
    }
}

// `f`, which touches no Python object, without the interpreter lock.
struct Unlocked {
    PyThreadState *state = PyEval_SaveThread();
    ~Unlocked() { PyEval_RestoreThread(state); }
};
template <typename F>
bool unlocked(F &&f) {
    const Unlocked here;
    return f();
}

PyObject *wrap(bool done, Tensor &y) { return done ? THPVariable_Wrap(std::move(y)) : none(); }

// linear(layer, x)
PyObject *py_linear(PyObject *, PyObject *const *args, Py_ssize_t n) {
    return guarded([&]() -> PyObject * {
        Tensor x, y;
        Linear l;
        if (n != 2 || !as_tensor(args[1], x) || !read_linear(args[0], l)) return none();
        return wrap(unlocked([&] { return product(x, l.p, l.bias, Flags(), y); }), y);
    });
}

// quantized_matmul(x, weight, scales, biases, quant, transpose, row_exact, rows, scratch, bias)
PyObject *py_quantized_matmul(PyObject *, PyObject *const *args, Py_ssize_t n) {
    return guarded([&]() -> PyObject * {
        Tensor x, bias, y;
        Packed p;
        if (n != 10 || !as_tensor(args[0], x) || !as_tensor(args[1], p.w) || !as_tensor(args[2], p.s) || !as_tensor(args[3], p.b) ||
            !read_quant(args[4], p.q) || !as_tensor(args[9], bias))
            return none();
        int flag[4];
        for (int i = 0; i < 4; i++)
            if ((flag[i] = PyObject_IsTrue(args[5 + i])) < 0) return nullptr;
        const Flags f{flag[0] != 0, flag[1] != 0, flag[2] != 0, flag[3] != 0};
        return wrap(unlocked([&] { return product(x, p, bias, f, y); }), y);
    });
}

// Whether `l` takes rows of `inner` values of `type` (the rest of `product`'s checks is x's).
bool linear_fits(const Linear &l, const Place &at, at::ScalarType type, int64_t inner) {
    int64_t columns;
    return l.p.fits(at, type, 2, columns) && columns == inner && bias_fits(l.bias, at, type, l.p.w.size(0));
}

// mlp(block, x): layers.Mlp.forward
PyObject *py_mlp(PyObject *, PyObject *const *args, Py_ssize_t n) {
    return guarded([&]() -> PyObject * {
        Tensor x, hidden, y;
        Linear down, gate, up, fused;
        if (n != 2 || !as_tensor(args[1], x) || !x.defined() || x.dim() < 1 || x.numel() == 0) return none();
        Ref geglu(PyObject_GetAttr(args[0], names.geglu)), both(PyObject_GetAttr(args[0], names.gate_up_proj));
        if (geglu.p == nullptr || both.p == nullptr || !read_linear(args[0], names.down_proj, down) ||
            !read_linear(args[0], names.gate_proj, gate)) {
            PyErr_Clear();
            return none();
        }
        const int truth = PyObject_IsTrue(geglu.p);
        if (truth < 0) return nullptr;
        const int32_t activation = truth ? NVQ_GLU_GEGLU : NVQ_GLU_SWIGLU;
        const int64_t rows = x.numel() / x.size(-1), most = gate.p.q.mode == NVQ_AFFINE ? 2 : 4;  // (layers.Mlp.forward says why)
        const Place at(x);
        const at::ScalarType type = x.scalar_type();
        if (!linear_fits(gate, at, type, x.size(-1)) || !linear_fits(down, at, type, gate.p.w.size(0))) return none();
        const bool several = rows > most;
        bool paired = both.p != Py_None;
        Several asked;
        if (paired && several) {  // (what the projections' sizes say already: the pair is not read where it would be refused)
            const nvq_qmm_desc d = gated_desc(x, code_of(type), gate.p.q, 2 * gate.p.w.size(0));
            asked.kernel = nvq_quantized_matmul_glu_several_takes(&d, &asked.need);
            paired = asked.kernel != 0;
        }
        if (paired) {
            const bool fits = read_linear(both.p, fused) && linear_fits(fused, at, type, x.size(-1)) && fused.p.w.size(0) == 2 * gate.p.w.size(0);
            if (!fits && !several) return none();
            if (fits) {
                const nvq_quant &q = gate.p.q, &r = fused.p.q;
                const bool same = q.mode == r.mode && q.group_size == r.group_size && q.bits == r.bits;
                const bool done = unlocked([&] {
                    return product_glu(x, fused.p, fused.bias, activation, 0.0f, 0.0f, several, same ? &asked : nullptr, hidden) && product(hidden, down.p, down.bias, Flags(), y);
                });
                if (hidden.defined()) return wrap(done, y);
            }
        }
        if (!read_linear(args[0], names.up_proj, up) || !linear_fits(up, at, type, x.size(-1)) || up.p.w.size(0) != gate.p.w.size(0)) return none();
        const bool done = unlocked([&] {
            Tensor g, u;
            return product(x, gate.p, gate.bias, Flags(), g) && product(x, up.p, up.bias, Flags(), u) && gated(g, u, activation, hidden) &&
                   product(hidden, down.p, down.bias, Flags(), y);
        });
        return wrap(done, y);
    });
}

bool read_projection(PyObject *o, PyObject *name, Projection &j) {
    Ref a(PyObject_GetAttr(o, name));
    if (a.p == nullptr) return declined();
    if (!projection_kind.plain(a.p)) return false;
    Tensor global_scale;
    if (!read_tensor(a.p, names.weight, j.p.w) || !read_tensor(a.p, names.scales, j.p.s) || !read_tensor(a.p, names.biases, j.p.b) ||
        !read_tensor(a.p, names.bias, j.bias) || !read_tensor(a.p, names.global_scale, global_scale) || global_scale.defined())
        return false;
    Ref q(PyObject_GetAttr(a.p, names.quant));
    return q.p == nullptr ? declined() : read_quant(q.p, j.p.q);
}

// moe(block, x): layers.MoeMlp.forward
PyObject *py_moe(PyObject *, PyObject *const *args, Py_ssize_t n) {
    return guarded([&]() -> PyObject * {
        Tensor x, router, y;
        int32_t k;
        bool normalize;
        Experts e;
        if (n != 2 || !moe_kind.plain(args[0]) || !as_tensor(args[1], x) || !read_tensor(args[0], names.gate, router) || !read_int(args[0], names.experts_per_token, k) ||
            !read_truth(args[0], names.norm_topk_prob, normalize))
            return none();
        Ref glu(PyObject_GetAttr(args[0], names.switch_mlp));
        if (glu.p == nullptr || !switch_glu_kind.plain(glu.p)) {
            PyErr_Clear();
            return none();
        }
        Ref both(PyObject_GetAttr(glu.p, names.gate_up_proj)), activation(PyObject_GetAttr(glu.p, names.activation));
        if (both.p == nullptr || activation.p == nullptr || !PyUnicode_Check(activation.p)) {
            PyErr_Clear();
            return none();
        }
        e.fused = both.p != Py_None;
        if (PyUnicode_CompareWithASCIIString(activation.p, "swiglu") == 0) e.act.code = NVQ_GLU_SWIGLU;
        else if (PyUnicode_CompareWithASCIIString(activation.p, "swiglu_oai") == 0) e.act.code = NVQ_GLU_SWIGLU_OAI;
        else if (PyUnicode_CompareWithASCIIString(activation.p, "geglu") == 0) e.act.code = NVQ_GLU_GEGLU;
        else return none();
        if (!read_projection(glu.p, names.gate_proj, e.gate) || !read_projection(glu.p, names.up_proj, e.up) ||
            !read_projection(glu.p, names.down_proj, e.down) || (e.fused && !read_projection(glu.p, names.gate_up_proj, e.both)) ||
            !read_truth(glu.p, names.gate_up_paired, e.paired) || !read_float(glu.p, names.alpha, e.act.alpha) ||
            !read_float(glu.p, names.limit, e.act.limit))
            return none();
        return wrap(unlocked([&] { return moe(x, router, k, normalize, e, y); }), y);
    });
}

// quantize(w, quant): (packed, scales, biases)
PyObject *py_quantize(PyObject *, PyObject *const *args, Py_ssize_t n) {
    return guarded([&]() -> PyObject * {
        Tensor w;
        nvq_quant q;
        if (n != 2 || !as_tensor(args[0], w) || !read_quant(args[1], q)) return none();
        const Place at(w);
        if (!at.usable() || w.dim() < 2 || w.numel() == 0 || !w.is_contiguous() || code_of(w.scalar_type()) < 0) return none();
        const int64_t cols = w.size(-1);
        if (q.group_size <= 0 || cols % q.group_size != 0) return none();
        const bool affine = q.mode == NVQ_AFFINE;
        const Sizes groups = with_last(w.sizes(), cols / q.group_size);
        Tensor packed, scales, biases;
        const bool done = unlocked([&] {
            packed = at.empty(with_last(w.sizes(), cols * q.bits / 32), at::kUInt32);
            scales = at.empty(groups, affine ? w.scalar_type() : at::kByte);
            if (affine) biases = at.empty(groups, w.scalar_type());
            return nvq_quantize(&q, code_of(w.scalar_type()), ptr(w), w.numel() / cols, cols, packed.mutable_data_ptr(), scales.mutable_data_ptr(),
                                affine ? biases.mutable_data_ptr() : nullptr, at.stream()) == NVQ_OK;
        });
        if (!done) return none();
        Ref p(THPVariable_Wrap(std::move(packed))), s(THPVariable_Wrap(std::move(scales)));
        Ref b(affine ? THPVariable_Wrap(std::move(biases)) : none());
        return p.p && s.p && b.p ? PyTuple_Pack(3, p.p, s.p, b.p) : nullptr;
    });
}

// The type a packed table gives its rows: the scales' for affine codes, else bfloat16 (ops.dequantize).
at::ScalarType table_type(const Packed &p) { return p.q.mode == NVQ_AFFINE && p.s.defined() ? p.s.scalar_type() : at::kBFloat16; }

bool is_dtype(PyObject *o, at::ScalarType &t) {
    if (!THPDtype_Check(o)) return false;
    t = reinterpret_cast<THPDtype *>(o)->scalar_type;
    return true;
}

// dequantize(weight, scales, biases, quant, dtype or None)
PyObject *py_dequantize(PyObject *, PyObject *const *args, Py_ssize_t n) {
    return guarded([&]() -> PyObject * {
        Packed p;
        if (n != 5 || !as_tensor(args[0], p.w) || !as_tensor(args[1], p.s) || !as_tensor(args[2], p.b) || !read_quant(args[3], p.q)) return none();
        const Place at(p.w);
        at::ScalarType type = table_type(p), asked = type;
        if (args[4] != Py_None && !is_dtype(args[4], asked)) return none();
        if (p.q.mode != NVQ_AFFINE) type = asked;
        int64_t columns;
        if (!at.usable() || code_of(type) < 0 || asked != type || p.w.dim() < 2 || p.w.numel() == 0 || !p.fits(at, type, p.w.dim(), columns))
            return none();
        Tensor y;
        const bool done = unlocked([&] {
            y = at.empty(with_last(p.w.sizes(), columns), type);
            return nvq_dequantize(&p.q, code_of(type), ptr(p.w), ptr(p.s), ptr(p.b), y.numel() / columns, columns, y.mutable_data_ptr(),
                                  at.stream()) == NVQ_OK;
        });
        return wrap(done, y);
    });
}

// embedding(weight, scales, biases, quant, ids)
PyObject *py_embedding(PyObject *, PyObject *const *args, Py_ssize_t n) {
    return guarded([&]() -> PyObject * {
        Packed p;
        Tensor ids;
        if (n != 5 || !as_tensor(args[0], p.w) || !as_tensor(args[1], p.s) || !as_tensor(args[2], p.b) || !read_quant(args[3], p.q) ||
            !as_tensor(args[4], ids))
            return none();
        const Place at(p.w);
        const at::ScalarType type = table_type(p);
        int64_t columns;
        if (!at.usable() || code_of(type) < 0 || !ids.defined() || !is_word(ids.scalar_type()) || !at.holds(ids) || ids.numel() == 0 ||
            !p.fits(at, type, 2, columns))
            return none();
        Sizes sizes(ids.sizes().begin(), ids.sizes().end());
        sizes.push_back(columns);
        Tensor y;
        const bool done = unlocked([&] {
            y = at.empty(sizes, type);
            return nvq_dequantize_rows(&p.q, code_of(type), ptr(p.w), ptr(p.s), ptr(p.b), p.w.size(0), columns, (const uint32_t *)ptr(ids),
                                       ids.numel(), y.mutable_data_ptr(), at.stream()) == NVQ_OK;
        });
        return wrap(done, y);
    });
}

// attention(q, k weight, scales, biases, v weight, scales, biases, quant, scale, sinks, causal[, several float32 rows too])
// (ops.quantized_attention, ops.quantized_attention_fits for one query row per head; ops.quantized_attention_prompt)
PyObject *py_attention(PyObject *, PyObject *const *args, Py_ssize_t n) {
    return guarded([&]() -> PyObject * {
        Tensor q, sinks;
        Packed k, v;
        if ((n != 11 && n != 12) || !as_tensor(args[0], q) || !as_tensor(args[1], k.w) || !as_tensor(args[2], k.s) || !as_tensor(args[3], k.b) ||
            !as_tensor(args[4], v.w) || !as_tensor(args[5], v.s) || !as_tensor(args[6], v.b) || !read_quant(args[7], k.q) ||
            !as_tensor(args[9], sinks))
            return none();
        v.q = k.q;
        const double scale = PyFloat_AsDouble(args[8]);
        if (scale == -1.0 && PyErr_Occurred()) {
            PyErr_Clear();
            return none();
        }
        const Place at(q);
        int64_t dim, same;
        if (!at.usable() || q.dim() != 4 || q.numel() == 0 || !q.is_contiguous() || k.q.mode != NVQ_AFFINE) return none();
        const at::ScalarType type = q.scalar_type();
        const int32_t code = code_of(type);
        if (code < 0 || !k.fits(at, type, 4, dim) || !v.fits(at, type, 4, same) || dim != q.size(3) || same != dim ||
            k.w.sizes() != v.w.sizes() || k.w.size(0) != q.size(0) || k.w.size(1) == 0 || k.w.size(2) == 0 ||
            !bias_fits(sinks, at, type, q.size(1)))
            return none();
        const nvq_attention_desc d{code, k.q.bits, k.q.group_size, (int32_t)dim, q.size(0), q.size(1), k.w.size(1), k.w.size(2), (float)scale};
        const bool several = q.size(2) > 1;
        // (ops.quantized_attention_fits: one query row takes caches of unsigned words)
        if (!several && (k.w.scalar_type() != at::kUInt32 || v.w.scalar_type() != at::kUInt32)) return none();
        const int causal = PyObject_IsTrue(args[10]), single_too = n == 12 ? PyObject_IsTrue(args[11]) : 0;
        if (causal < 0 || single_too < 0) return nullptr;
        const bool single = several && code == NVQ_F32;
        if (single && !single_too) return none();
        const nvq_attention_prompt_desc prompt{d, q.size(2), causal};
        Tensor y;
        const bool done = unlocked([&] {
            const size_t need = single    ? nvq_quantized_attention_prompt_f32_workspace_bytes(&prompt)
                                : several ? nvq_quantized_attention_prompt_workspace_bytes(&prompt)
                                          : nvq_quantized_attention_workspace_bytes(&d);
            if (several && !single && need == 0) return false;
            y = at.empty(q.sizes(), type);
            Tensor workspace;
            if (need > 0) workspace = at.empty({(int64_t)need}, at::kByte);
            void *scratch = need > 0 ? workspace.mutable_data_ptr() : nullptr;
            if (single)
                return nvq_quantized_attention_prompt_f32(&prompt, ptr(q), ptr(k.w), ptr(k.s), ptr(k.b), ptr(v.w), ptr(v.s), ptr(v.b), ptr(sinks),
                                                          y.mutable_data_ptr(), scratch, at.stream()) == NVQ_OK;
            return (several ? nvq_quantized_attention_prompt(&prompt, ptr(q), ptr(k.w), ptr(k.s), ptr(k.b), ptr(v.w), ptr(v.s), ptr(v.b), ptr(sinks),
                                                             y.mutable_data_ptr(), scratch, at.stream())
                            : nvq_quantized_attention(&d, ptr(q), ptr(k.w), ptr(k.s), ptr(k.b), ptr(v.w), ptr(v.s), ptr(v.b), ptr(sinks),
                                                      y.mutable_data_ptr(), scratch, at.stream())) == NVQ_OK;
        });
        return wrap(done, y);
    });
}

// register((type, {name: function}), ...): QuantizedLinear, SwitchProjection, SwitchGlu and MoeMlp with their own methods
PyObject *py_register(PyObject *, PyObject *const *args, Py_ssize_t n) {
    Kind *const kinds[] = {&linear_kind, &projection_kind, &switch_glu_kind, &moe_kind};
    PyObject *types[4], *methods[4];
    for (Py_ssize_t i = 0; i < 4; i++) {
        if (n != 4 || !PyArg_ParseTuple(args[i], "O!O!", &PyType_Type, &types[i], &PyDict_Type, &methods[i])) {
            PyErr_SetString(PyExc_TypeError, "register: four pairs of a class and its methods");
            return nullptr;
        }
    }
    for (Py_ssize_t i = 0; i < 4; i++) {
        Py_INCREF(types[i]), Py_INCREF(methods[i]);  // (kept until the process ends, with the names and functions they hold)
        kinds[i]->methods.clear();
        PyObject *name, *function;
        for (Py_ssize_t at = 0; PyDict_Next(methods[i], &at, &name, &function);) kinds[i]->methods.emplace_back(name, function);
        kinds[i]->type = (PyTypeObject *)types[i];
    }
    return none();
}

// ready(index): nvq_init has answered for the device
PyObject *py_ready(PyObject *, PyObject *index) {
    const long i = PyLong_AsLong(index);
    if (i == -1 && PyErr_Occurred()) return nullptr;
    if (i >= 0 && i < 64) ready_devices |= 1ull << i;
    return none();
}

#define NVQ_FAST(f) (PyCFunction)(void (*)(void)) f, METH_FASTCALL
PyMethodDef methods[] = {
    {"register", NVQ_FAST(py_register), nullptr},
    {"ready", py_ready, METH_O, nullptr},
    {"linear", NVQ_FAST(py_linear), nullptr},
    {"quantized_matmul", NVQ_FAST(py_quantized_matmul), nullptr},
    {"mlp", NVQ_FAST(py_mlp), nullptr},
    {"moe", NVQ_FAST(py_moe), nullptr},
    {"quantize", NVQ_FAST(py_quantize), nullptr},
    {"dequantize", NVQ_FAST(py_dequantize), nullptr},
    {"embedding", NVQ_FAST(py_embedding), nullptr},
    {"attention", NVQ_FAST(py_attention), nullptr},
    {nullptr, nullptr, 0, nullptr},
};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_native", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

extern "C" __attribute__((visibility("default"))) PyObject *PyInit__native(void) {
    struct { PyObject **at; const char *text; } all[] = {
        {&names.mode, "mode"}, {&names.group_size, "group_size"}, {&names.bits, "bits"}, {&names.weight, "weight"},
        {&names.scales, "scales"}, {&names.biases, "biases"}, {&names.bias, "bias"}, {&names.quant, "quant"},
        {&names.global_scale, "global_scale"}, {&names.gate_proj, "gate_proj"}, {&names.up_proj, "up_proj"},
        {&names.down_proj, "down_proj"}, {&names.gate_up_proj, "gate_up_proj"}, {&names.geglu, "geglu"},
        {&names.gate, "gate"}, {&names.switch_mlp, "switch_mlp"}, {&names.experts_per_token, "experts_per_token"},
        {&names.norm_topk_prob, "norm_topk_prob"}, {&names.gate_up_paired, "gate_up_paired"}, {&names.activation, "activation"},
        {&names.alpha, "alpha"}, {&names.limit, "limit"},
    };
    for (auto &n : all) {
        *n.at = PyUnicode_InternFromString(n.text);
        if (*n.at == nullptr) return nullptr;
    }
    return PyModule_Create(&module);
}
