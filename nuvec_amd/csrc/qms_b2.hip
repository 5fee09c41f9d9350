// The split-K kernel of a few dozen rows for affine 2-bit codes (qms_kernel.h).
#include "qms_kernel.h"

namespace nvq {
int32_t launch_qms_b2(const ProductArgs &a, const qms::Plan &p, hipStream_t s) { return qms::run_dtype<2, qmf::kAffine>(a, p, s); }
}  // namespace nvq
