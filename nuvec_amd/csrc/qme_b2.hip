// The grouped kernel of sorted pairs for affine 2-bit codes (qme_kernel.h).
#include "qme_kernel.h"

namespace nvq {
int32_t launch_qme_b2(const ProductArgs &a, hipStream_t s) { return qme::run_dtype<2, rows::kAffine>(a, s); }
}  // namespace nvq
