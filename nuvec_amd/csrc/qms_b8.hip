// The split-K kernel of a few dozen rows for affine 8-bit codes (qms_kernel.h).
#include "qms_kernel.h"

namespace nvq {
int32_t launch_qms_b8(const ProductArgs &a, const qms::Plan &p, hipStream_t s) { return qms::run_dtype<8, qmf::kAffine>(a, p, s); }
}  // namespace nvq
