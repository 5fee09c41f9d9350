// The few-row and tiled matrix-core kernels for NVFP4 codes (a global scale folded into the group scales) (qmf_kernel.h,
// qmm_kernel.h).
#include "qmf_kernel.h"
#include "qmk_kernel.h"

namespace nvq {

int32_t launch_qmf_nvfp4(const ProductArgs &a, hipStream_t s) {
    return qmf::run_dtype<4, qmf::kNvfp4>(a, s);
}

int32_t launch_qmm_nvfp4(const ProductArgs &a, void *workspace, hipStream_t s) { return run_tiled<4, qmf::kNvfp4>(a, workspace, s); }

}  // namespace nvq
