// The few-row and tiled matrix-core kernels for affine 8-bit codes (qmf_kernel.h, qmm_kernel.h).
#include "qmf_kernel.h"
#include "qmk_kernel.h"

namespace nvq {

int32_t launch_qmf_b8(const ProductArgs &a, hipStream_t s) { return qmf::run_dtype<8, false>(a, s); }

int32_t launch_qmm_b8(const ProductArgs &a, void *workspace, hipStream_t s) { return run_tiled<8, false>(a, workspace, s); }

}  // namespace nvq
