// Routing of the few-row and the grouped matrix-core kernels (qmf_kernel.h, qme_kernel.h, qmg_kernel.h): which products
// they take and the per-width entry points.
#include "qmg_kernel.h"

#include <math.h>

namespace nvq {

// The grouped kernel: one row of x per pair, its scale table within its LDS budget, K of whole steps of 64
// (windows of 128 for 1, 3 and 5 bits) or, beyond one window, whole 32 values (not with a global scale, whose weights the
// element type does not hold).  Row-exact pairs keep the vector kernels where they had them, with the
// CPU's weights and off whole steps.
static bool grouped_supported(const ProductArgs &a) {
    if (a.m != 1 || a.experts > 65535) return false;
    const bool odd = a.mode == NVQ_AFFINE && a.bits % 2 != 0, whole = a.k >= 64 && a.k % (odd ? 128 : 64) == 0;
    if (a.row_exact && (a.exact_weights || !whole)) return false;
    if (whole ? qmg::table_bytes(a) > (size_t)qmg::kTableMaxBytes : qmg::lds_bytes(a) > (size_t)qmg::kLdsMost) return false;
    return whole || (a.k >= 128 && a.k % 32 == 0 && (a.mode == NVQ_AFFINE || a.global_scale == nullptr));
}

// The rows of one product as one group: affine codes off whole steps of 64 whose weights are not the CPU's (those are the tiled
// kernel's).  The vector kernel's passes of four rows take 1 us per 2.1 M weights, a window of this kernel 2.5 us with one
// or two blocks on a compute unit.
bool grouped_rows_take(const ProductArgs &a) {
    if ((a.dtype != NVQ_BF16 && a.dtype != NVQ_F16) || a.mode != NVQ_AFFINE || a.exact_weights || a.row_exact || a.batch != 1 || a.batch_ndim != 0 ||
        a.rhs != nullptr || a.lhs != nullptr || a.glu != 0 || a.k % 64 != 32 || a.k < 128 || qmg::lds_bytes(a) > (size_t)qmg::kLdsMost)
        return false;
    const double blocks = (double)((a.n + qmg::kRows - 1) / qmg::kRows) * (double)((a.m + qmg::kPassRows - 1) / qmg::kPassRows);
    if (blocks > 1e8) return false;
    const double per_unit = qmg::lds_bytes(a) <= (size_t)qmg::kLdsMost / 2 ? 2.0 : 1.0;
    const double here = 15.0 + ceil(blocks / (per_unit * fmax(1.0, (double)compute_units()))) * (double)((a.k + 127) / 128) * 2.5;
    return here < 0.8 * (double)((a.m + 3) / 4) * (double)a.n * (double)a.k / 2.1e6;
}

int32_t launch_grouped_rows(ProductArgs a, hipStream_t s) {
    a.one_group = 1, a.experts = 1;
    a.batch = a.x_batches = a.m, a.m = 1;
    a.expert_bias = a.row_bias, a.row_bias = nullptr;
    return launch_qmf(a, s);
}

// Whether the few-row matrix-core kernel takes this product: a block format or affine 1 to 6 or 8 bits, bf16 or
// f16, whole steps of 64 values (whole windows of 128 for 1, 3 and 5 bits, whose 16-byte chunks straddle steps),
// a scale table that fits in LDS, and either no batch, a batch with one stride per operand, gathered pairs,
// or the grouped gather.
bool qmf_supported(const ProductArgs &a) {
    if (a.dtype != NVQ_BF16 && a.dtype != NVQ_F16) return false;
    if (a.offsets != nullptr) return grouped_supported(a);
    if (a.k < 64 || a.k % 64 != 0) return false;
    size_t lds = 0;
    if (a.mode == NVQ_MXFP4 || a.mode == NVQ_NVFP4) {
        lds = qmf::lds_needed<4>(a);
    } else if (a.mode == NVQ_MXFP8) {
        lds = qmf::lds_needed<8>(a);
    } else if (a.mode == NVQ_AFFINE) {
        switch (a.bits) {
        case 1: lds = qmf::lds_needed<1>(a); break;
        case 2: lds = qmf::lds_needed<2>(a); break;
        case 3: lds = qmf::lds_needed<3>(a); break;
        case 4: lds = qmf::lds_needed<4>(a); break;
        case 5: lds = qmf::lds_needed<5>(a); break;
        case 6: lds = qmf::lds_needed<6>(a); break;
        case 8: lds = qmf::lds_needed<8>(a); break;
        default: return false;
        }
        if (a.bits % 2 != 0 && a.k % 128 != 0) return false;
    } else {
        return false;
    }
    if (lds > (size_t)qmf::kLdsLimit) return false;
    if (a.rhs != nullptr) return a.batch <= 65535 && (a.m + 31) / 32 <= 65535;  // gathered pairs, one per grid z
    return (a.batch == 1 || a.batch_ndim == 1) && a.batch <= 65535 && (a.m + 31) / 32 <= 65535;
}

// Sorted pairs whose weights the kernel holds in the element type; affine ones off whole steps that are not the CPU's stay with
// qmg_kernel's terms.
static int32_t launch_qme(const ProductArgs &a, hipStream_t s) {
    if (a.mode == NVQ_MXFP4) return launch_qme_fp4(a, s);
    if (a.mode == NVQ_MXFP8) return launch_qme_fp8(a, s);
    if (a.mode == NVQ_NVFP4) return launch_qme_nvfp4(a, s);
    switch (a.bits) {
    case 1: return launch_qme_b1(a, s);
    case 2: return launch_qme_b2(a, s);
    case 3: return launch_qme_b3(a, s);
    case 4: return launch_qme_b4(a, s);
    case 5: return launch_qme_b5(a, s);
    case 6: return launch_qme_b6(a, s);
    default: return launch_qme_b8(a, s);
    }
}

int32_t launch_qmf(const ProductArgs &a, hipStream_t s) {
    if (a.offsets != nullptr && (a.mode != NVQ_AFFINE || a.exact_weights || a.k % (a.bits % 2 != 0 ? 128 : 64) == 0)) return launch_qme(a, s);
    if (a.mode == NVQ_MXFP4) return launch_qmf_fp4(a, s);
    if (a.mode == NVQ_MXFP8) return launch_qmf_fp8(a, s);
    if (a.mode == NVQ_NVFP4) return launch_qmf_nvfp4(a, s);
    switch (a.bits) {
    case 1: return launch_qmf_b1(a, s);
    case 2: return launch_qmf_b2(a, s);
    case 3: return launch_qmf_b3(a, s);
    case 4: return launch_qmf_b4(a, s);
    case 5: return launch_qmf_b5(a, s);
    case 6: return launch_qmf_b6(a, s);
    default: return launch_qmf_b8(a, s);
    }
}

}  // namespace nvq
