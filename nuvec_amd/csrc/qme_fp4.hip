// The grouped kernel of sorted pairs for MXFP4 codes (qme_kernel.h).
#include "qme_kernel.h"

namespace nvq {
int32_t launch_qme_fp4(const ProductArgs &a, hipStream_t s) { return qme::run_dtype<4, rows::kMxfp4>(a, s); }
}  // namespace nvq
