// The grouped kernel of sorted pairs for affine 6-bit codes (qmg_kernel.h).
#include "qmg_kernel.h"

namespace nvq {
int32_t launch_qmg_b6(const ProductArgs &a, hipStream_t s) { return qmg::run_dtype<6, rows::kAffine>(a, s); }
}  // namespace nvq
