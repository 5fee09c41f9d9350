// The grouped kernel of sorted pairs for affine 4-bit codes (qme_kernel.h).
#include "qme_kernel.h"

namespace nvq {
int32_t launch_qme_b4(const ProductArgs &a, hipStream_t s) { return qme::run_dtype<4, rows::kAffine>(a, s); }
}  // namespace nvq
