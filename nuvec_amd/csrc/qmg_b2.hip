// The grouped kernel of sorted pairs for affine 2-bit codes (qmg_kernel.h).
#include "qmg_kernel.h"

namespace nvq {
int32_t launch_qmg_b2(const ProductArgs &a, hipStream_t s) { return qmg::run_dtype<2, rows::kAffine>(a, s); }
}  // namespace nvq
