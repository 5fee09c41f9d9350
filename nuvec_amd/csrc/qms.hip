// How the split-K kernel of a few dozen rows (qms_kernel.h) cuts a product, and which products it takes.
#include "qms_kernel.h"

#include <math.h>

namespace nvq {

// One product (no batch, no gathered pairs, not row-exact) in bfloat16 or float16 against weights stored [N, K].
static bool qms_supported(const ProductArgs &a) {
    if (a.dtype == NVQ_F32 || a.row_exact || a.batch != 1 || a.batch_ndim != 0 || a.rhs != nullptr || a.lhs != nullptr || a.offsets != nullptr) return false;
    if (a.mode == NVQ_AFFINE && (a.bits == 1 || (a.group != 32 && a.group != 64 && a.group != 128))) return false;
    if (a.k < 32 || a.k % 32 != 0 || a.k / 32 * a.bits < 4 || a.k > 1 << 26) return false;  // (a chunk of codes lies inside a row)
    if (a.glu != 0 && (a.n % 128 != 0 || a.exact_weights)) return false;
    return a.m >= 1 && (a.m + 15) / 16 <= 65535 && a.n >= 1 && a.n <= 0x7FFFFFFF / 64 && ((uintptr_t)a.x | (uintptr_t)a.w) % 16 == 0;
}

// The cut with the least estimated time.  A turn of 256 values takes a wavefront about a microsecond per tile of weight rows, whatever is
// beside it on its SIMD; a split adds a second kernel and its traffic.  Fitted (16 % off on average) to 35000 timings of 1248 products
// of 3 to 400 rows, 18 weight shapes from W[640,1088] to W[27136,2112] and W[2560,11072], six affine formats and the three block
// formats; choosing by it is 2 % above always taking the fastest cut.  The parts fit the library's own scratch.
bool qms_plan(const ProductArgs &a, qms::Plan &best) {
    if (!qms_supported(a)) return false;
    best = qms::Plan{};
    const int64_t tiles = (a.m + 15) / 16, spans = (a.k + qms::kSpan - 1) / qms::kSpan;
    const int mt = tiles == 1 ? 1 : tiles == 2 ? 2 : 4;
    const double cus = fmax(1.0, (double)compute_units()), passes = (double)((tiles + mt - 1) / mt), outputs = (double)a.m * (double)a.n;
    const double format = a.mode == NVQ_MXFP4 || a.mode == NVQ_MXFP8 ? 0.74 : 1.0;
    struct Cut { int nt, qw, groups; };
    static const Cut cuts[] = {{1, 4, 1}, {1, 4, 2}, {2, 4, 1}, {2, 4, 2}, {1, 1, 2}, {1, 1, 4}, {1, 1, 8}, {1, 1, 16}, {2, 1, 2}, {2, 1, 4}, {2, 1, 8}, {2, 1, 16}};
    for (const Cut &c : cuts) {
        if (!qms::has_shape(mt, c.nt, c.qw) || c.groups > qms::most_groups(mt, c.nt, c.qw) || c.groups > spans || (a.glu != 0 && c.nt != 2)) continue;
        if (c.groups > 1 && qms::lds_bytes(a.bits, mt, c.nt, c.qw, c.groups) > 160 * 1024) continue;
        const double tile_blocks = passes * (double)((a.n + 64 * c.nt - 1) / (64 * c.nt) * (4 / c.qw));
        const double turn_us = format * (1.06 * c.nt + 0.12 * mt + 0.07 * mt * c.nt - 0.04);
        static const int counts[] = {1, 2, 3, 4, 6, 8, 12, 16};
        for (const int want : counts) {
            if (want > spans || (c.qw == 1 && want > 4) || (want > 1 && (double)want * outputs * 4.0 > (double)NVQ_STATIC_SCRATCH_BYTES)) break;
            const int64_t per = (spans + want - 1) / want, splits = (spans + per - 1) / per, turns = (per + c.groups - 1) / c.groups;
            const double load = fmax(1.0, ceil(tile_blocks * (double)splits / cus) * (double)(c.groups * c.qw) / 4.0 * 0.81);
            const double us = 3.7 + (double)turns * turn_us * load + (splits > 1 ? 2.8 + 1.5e-6 * (double)splits * outputs : 0.0);
            if (best.mt == 0 || us < best.us) best = qms::Plan{mt, c.nt, c.qw, c.groups, (int)splits, (int)per, us};
        }
    }
    return best.mt != 0;
}

size_t qms_workspace_bytes(const ProductArgs &a, const qms::Plan &p) {
    return p.splits > 1 ? (size_t)p.splits * (size_t)a.m * (size_t)a.n * sizeof(float) : 0;
}

const char *qms_kernel_name(const qms::Plan &p) {
    switch (100 * p.mt + 10 * p.nt + p.qw) {
    case 111: return "qms_kernel<1,1,1>";
    case 121: return "qms_kernel<1,2,1>";
    case 114: return "qms_kernel<1,1,4>";
    case 211: return "qms_kernel<2,1,1>";
    case 214: return "qms_kernel<2,1,4>";
    case 224: return "qms_kernel<2,2,4>";
    case 414: return "qms_kernel<4,1,4>";
    default: return "qms_kernel<4,2,4>";
    }
}

int32_t launch_qms(const ProductArgs &args, const qms::Plan &p, void *workspace, hipStream_t s) {
    ProductArgs a = args;
    a.k_splits = workspace != nullptr ? p.splits : 1;
    a.k_split_steps = p.spans;
    a.partials = (float *)workspace;
    if (a.mode == NVQ_MXFP4) return launch_qms_fp4(a, p, s);
    if (a.mode == NVQ_MXFP8) return launch_qms_fp8(a, p, s);
    if (a.mode == NVQ_NVFP4) return launch_qms_nvfp4(a, p, s);
    switch (a.bits) {
    case 2: return launch_qms_b2(a, p, s);
    case 3: return launch_qms_b3(a, p, s);
    case 4: return launch_qms_b4(a, p, s);
    case 5: return launch_qms_b5(a, p, s);
    case 6: return launch_qms_b6(a, p, s);
    default: return launch_qms_b8(a, p, s);
    }
}

}  // namespace nvq
