// Reductions over a wavefront on the vector unit alone.
#pragma once
#include "nvq_device.h"

namespace nvq {
namespace {

// v + (v moved across lanes by a DPP control); lanes the control does not feed add 0.
template <int CTRL, int ROW_MASK>
__device__ __forceinline__ float dpp_add(float v) {
    const int moved = __builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, ROW_MASK, 0xF, true);
    return v + __int_as_float(moved);
}

// Sum over the wavefront in VALU data-parallel-primitive steps (no LDS traffic): shifts by
// 1, 2, 4, 8 inside each row of 16 lanes, then the row totals carried into the next rows.
// The total is valid in lane 63 only.
__device__ __forceinline__ float wave_sum_lane63(float v) {
    v = dpp_add<0x111, 0xF>(v);  // row_shr:1
    v = dpp_add<0x112, 0xF>(v);  // row_shr:2
    v = dpp_add<0x114, 0xF>(v);  // row_shr:4
    v = dpp_add<0x118, 0xF>(v);  // row_shr:8
    v = dpp_add<0x142, 0xA>(v);  // row_bcast:15 into rows 1 and 3
    v = dpp_add<0x143, 0xC>(v);  // row_bcast:31 into rows 2 and 3
    return v;
}

// The maximum likewise (lanes the control does not feed keep theirs), as fmaxf has it; valid in lane 63 only.
template <int CTRL, int ROW_MASK>
__device__ __forceinline__ float dpp_max(float v) {
    const int own = __float_as_int(v);
    return fmaxf(v, __int_as_float(__builtin_amdgcn_update_dpp(own, own, CTRL, ROW_MASK, 0xF, false)));
}
__device__ __forceinline__ float wave_max_lane63(float v) {
    v = dpp_max<0x111, 0xF>(v);
    v = dpp_max<0x112, 0xF>(v);
    v = dpp_max<0x114, 0xF>(v);
    v = dpp_max<0x118, 0xF>(v);
    v = dpp_max<0x142, 0xA>(v);
    return dpp_max<0x143, 0xC>(v);
}
__device__ __forceinline__ float from_lane(float v, int lane) { return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), lane)); }

}  // namespace
}  // namespace nvq
