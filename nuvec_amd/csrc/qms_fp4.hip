// The split-K kernel of a few dozen rows for MXFP4 codes (qms_kernel.h).
#include "qms_kernel.h"

namespace nvq {
int32_t launch_qms_fp4(const ProductArgs &a, const qms::Plan &p, hipStream_t s) { return qms::run_dtype<4, qmf::kMxfp4>(a, p, s); }
}  // namespace nvq
