// The grouped kernel of sorted pairs for NVFP4 codes (qme_kernel.h).
#include "qme_kernel.h"

namespace nvq {
int32_t launch_qme_nvfp4(const ProductArgs &a, hipStream_t s) { return qme::run_dtype<4, rows::kNvfp4>(a, s); }
}  // namespace nvq
