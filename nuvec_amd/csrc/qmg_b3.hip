// The grouped kernel of sorted pairs for affine 3-bit codes (qmg_kernel.h).
#include "qmg_kernel.h"

namespace nvq {
int32_t launch_qmg_b3(const ProductArgs &a, hipStream_t s) { return qmg::run_dtype<3, rows::kAffine>(a, s); }
}  // namespace nvq
