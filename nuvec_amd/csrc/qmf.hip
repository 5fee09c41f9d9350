// Routing of the few-row and the grouped matrix-core kernels (qmf_kernel.h, qmg_kernel.h): which products they take and the per-width
// entry points.
#include "qmf_kernel.h"

#include <math.h>

namespace nvq {

// The grouped kernel: one row of x per pair, K of whole steps of 64 (windows of 128 for 1, 3 and 5 bits) or, beyond one window, whole 32
// values (not with a global scale, whose weights the element type does not hold).  Row-exact pairs keep the vector kernels where they
// had them, with the CPU's weights and off whole steps.
static bool grouped_supported(const ProductArgs &a) {
    if (a.m != 1 || a.experts > 65535) return false;
    const bool odd = a.mode == NVQ_AFFINE && a.bits % 2 != 0, whole = a.k >= 64 && a.k % (odd ? 128 : 64) == 0;
    if (a.row_exact && (a.exact_weights || !whole)) return false;
    return whole || (a.k >= 128 && a.k % 32 == 0 && (a.mode == NVQ_AFFINE || a.global_scale == nullptr));
}

// The rows of one product as one group: affine codes off whole steps of 64 whose weights are not the CPU's (those are the tiled
// kernel's).  A window takes this kernel 1.6 us with up to two blocks on a compute unit, a pass of four rows the vector kernel 1 us per
// 1.8 M weights: 107 products of 2 to 700 rows timed on both, 1.2 % above always taking the faster one, 1.62 x at worst.
bool grouped_rows_take(const ProductArgs &a) {
    if ((a.dtype != NVQ_BF16 && a.dtype != NVQ_F16) || a.mode != NVQ_AFFINE || a.exact_weights || a.row_exact || a.batch != 1 || a.batch_ndim != 0 ||
        a.rhs != nullptr || a.lhs != nullptr || a.glu != 0 || a.k % 64 != 32 || a.k < 128)
        return false;
    const double blocks = (double)((a.n + 127) / 128) * (double)((a.m + 63) / 64);
    if (blocks > 1e8) return false;
    const double here = 4.0 + ceil(blocks / (2.0 * fmax(1.0, (double)compute_units()))) * (double)((a.k + 127) / 128) * 1.6;
    return here < (double)((a.m + 3) / 4) * (double)a.n * (double)a.k / 1.8e6;
}

int32_t launch_grouped_rows(ProductArgs a, hipStream_t s) {
    a.one_group = 1, a.experts = 1;
    a.batch = a.x_batches = a.m, a.m = 1;
    a.expert_bias = a.row_bias, a.row_bias = nullptr;
    return launch_qmf(a, s);
}

// The gate and up products of several rows as the one group of the grouped kernel, with the gated activation as its epilogue, and the
// groups of a block that are estimated fastest.  A compute unit works off its blocks' windows at a rate (thr), a wavefront its own chain
// of them no faster than at another (lat), four groups of wavefronts at a time.  Fitted to 20000 timings of 6900 pairs of 6 to 512 rows, K
// 512 to 5120, 2560 to 14336 hidden values, twelve formats, with one, two and four groups: 12 % off on average, and the groups chosen by it
// are 2 % above the fastest.  Every call pays for the choice (host, 8 rows of a refused [1024,512] pair 0.38 us with all nine powers and the
// cuts walked for each question, 0.11 so): no powers are taken for a number of groups whose rates alone are beyond `most` or the best so far.
double gated_group_us(const ProductArgs &a, double most, int &groups) {
    groups = 1;
    const bool odd = a.mode == NVQ_AFFINE && a.bits % 2 != 0;
    if ((a.dtype != NVQ_BF16 && a.dtype != NVQ_F16) || (a.mode == NVQ_AFFINE && a.bits == 1) || a.exact_weights || a.global_scale != nullptr || a.k < 128 ||
        a.k % (odd ? 128 : 64) != 0 || a.n % 128 != 0 || a.n > 0x7FFFFFFF || a.m < 1 || a.m > 256)
        return HUGE_VAL;
    const double format = a.mode == NVQ_MXFP4 ? 0.76 : a.mode == NVQ_MXFP8 ? 1.05 : a.mode == NVQ_NVFP4 ? 1.03 : a.bits == 2 ? 1.0 : a.bits == 3 ? 1.07
                          : a.bits == 4 ? 1.04 : a.bits == 5 ? 1.22 : a.bits == 6 ? 1.24 : 1.29;
    const int64_t passes = (a.m + 63) / 64, windows = (a.k + 127) / 128;
    const double tiles = (double)((a.m + 15) / 16) / (double)passes;  // of 16 rows, of a pass
    const double blocks = ceil((double)(a.n / 128 * passes) / fmax(1.0, (double)compute_units()));  // of a compute unit
    double best = most;
    for (int g = 1; g <= 4 && g <= windows; g *= 2) {
        const double turns = (double)((windows + g - 1) / g), around = 2.9 + 0.51 * (g - 1) + 2.68 * blocks;
        const double thr = blocks * g * turns * format * (0.467 + 0.119 * tiles);
        const double lat = ceil(blocks * g / 4.0) * turns * (0.52 + 0.231 * tiles);  // times format^1.15, no less than 0.95 of it
        if (!(around + fmax(thr, 0.95 * format * lat) < best)) continue;
        const double us = around + pow(pow(thr, 2.65) + pow(pow(format, 1.15) * lat, 2.65), 1.0 / 2.65);
        if (us < best) best = us, groups = g;
    }
    return best < most ? best : HUGE_VAL;
}

int32_t launch_gated_group(ProductArgs a, int groups, hipStream_t s) {
    a.k_splits = groups;
    return launch_grouped_rows(a, s);
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

static int32_t launch_grouped(const ProductArgs &a, hipStream_t s) {
    if (a.mode == NVQ_MXFP4) return launch_qmg_fp4(a, s);
    if (a.mode == NVQ_MXFP8) return launch_qmg_fp8(a, s);
    if (a.mode == NVQ_NVFP4) return launch_qmg_nvfp4(a, s);
    switch (a.bits) {
    case 1: return launch_qmg_b1(a, s);
    case 2: return launch_qmg_b2(a, s);
    case 3: return launch_qmg_b3(a, s);
    case 4: return launch_qmg_b4(a, s);
    case 5: return launch_qmg_b5(a, s);
    case 6: return launch_qmg_b6(a, s);
    default: return launch_qmg_b8(a, s);
    }
}

int32_t launch_qmf(const ProductArgs &a, hipStream_t s) {
    if (a.offsets != nullptr || a.one_group) return launch_grouped(a, s);
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
