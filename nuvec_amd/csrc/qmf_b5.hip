// The few-row and tiled matrix-core kernels for affine 5-bit codes (qmf_kernel.h, qmm_kernel.h).
#include "qmf_kernel.h"
#include "qmk_kernel.h"

namespace nvq {

int32_t launch_qmf_b5(const ProductArgs &a, hipStream_t s) { return qmf::run_dtype<5, false>(a, s); }

int32_t launch_qmm_b5(const ProductArgs &a, void *workspace, hipStream_t s) { return run_tiled<5, false>(a, workspace, s); }

}  // namespace nvq
