// The split-K kernel of a few dozen rows for MXFP8 codes (qms_kernel.h).
#include "qms_kernel.h"

namespace nvq {
int32_t launch_qms_fp8(const ProductArgs &a, const qms::Plan &p, hipStream_t s) { return qms::run_dtype<8, qmf::kMxfp8>(a, p, s); }
}  // namespace nvq
