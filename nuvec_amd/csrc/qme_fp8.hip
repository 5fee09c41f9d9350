// The grouped kernel of sorted pairs for MXFP8 codes (qme_kernel.h).
#include "qme_kernel.h"

namespace nvq {
int32_t launch_qme_fp8(const ProductArgs &a, hipStream_t s) { return qme::run_dtype<8, rows::kMxfp8>(a, s); }
}  // namespace nvq
