// The grouped kernel of sorted pairs for affine 5-bit codes (qmg_kernel.h).
#include "qmg_kernel.h"

namespace nvq {
int32_t launch_qmg_b5(const ProductArgs &a, hipStream_t s) { return qmg::run_dtype<5, rows::kAffine>(a, s); }
}  // namespace nvq
