// The grouped kernel of sorted pairs for MXFP4 codes (qmg_kernel.h).
#include "qmg_kernel.h"

namespace nvq {
int32_t launch_qmg_fp4(const ProductArgs &a, hipStream_t s) { return qmg::run_dtype<4, rows::kMxfp4>(a, s); }
}  // namespace nvq
