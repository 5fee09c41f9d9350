// The few-row and tiled matrix-core kernels for MXFP4 codes (qmf_kernel.h, qmm_kernel.h).
#include "qmf_kernel.h"
#include "qmk_kernel.h"

namespace nvq {

int32_t launch_qmf_fp4(const ProductArgs &a, hipStream_t s) {
    return qmf::run_dtype<4, true>(a, s);
}

int32_t launch_qmm_fp4(const ProductArgs &a, void *workspace, hipStream_t s) { return run_tiled<4, true>(a, workspace, s); }

}  // namespace nvq
