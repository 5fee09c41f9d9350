// The grouped kernel of sorted pairs for MXFP8 codes (qmg_kernel.h).
#include "qmg_kernel.h"

namespace nvq {
int32_t launch_qmg_fp8(const ProductArgs &a, hipStream_t s) { return qmg::run_dtype<8, rows::kMxfp8>(a, s); }
}  // namespace nvq
