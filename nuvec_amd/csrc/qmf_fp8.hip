// The few-row and tiled matrix-core kernels for MXFP8 codes (qmf_kernel.h, qmm_kernel.h).
#include "qmf_kernel.h"
#include "qmk_kernel.h"

namespace nvq {

int32_t launch_qmf_fp8(const ProductArgs &a, hipStream_t s) {
    return qmf::run_dtype<8, qmf::kMxfp8>(a, s);
}

int32_t launch_qmm_fp8(const ProductArgs &a, void *workspace, hipStream_t s) { return run_tiled<8, qmf::kMxfp8>(a, workspace, s); }

}  // namespace nvq
