// wave_dpp.hpp -- sums over a wave by DPP lane shifts, in a fixed order.
#pragma once

#include "internal.hpp"

namespace mtl4g {

// v of another lane of the wave by DPP, 0 where the row mask or the row's edge
// leaves a lane without a source.
template <int CTRL, int ROWS>
__device__ __forceinline__ double res_dpp(double v) {
    const unsigned long long b = (unsigned long long)__double_as_longlong(v);
    const unsigned lo = (unsigned)__builtin_amdgcn_update_dpp(0, (int)(unsigned)b, CTRL, ROWS, 0xf, true);
    const unsigned hi = (unsigned)__builtin_amdgcn_update_dpp(0, (int)(unsigned)(b >> 32), CTRL, ROWS, 0xf, true);
    return __longlong_as_double((long long)(((unsigned long long)hi << 32) | lo));
}
template <int CTRL, int ROWS>
__device__ __forceinline__ float res_dpp(float v) {
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, ROWS, 0xf, true));
}
__device__ __forceinline__ double res_lane(double v, int lane) {
    const unsigned long long b = (unsigned long long)__double_as_longlong(v);
    const unsigned lo = (unsigned)__builtin_amdgcn_readlane((int)(unsigned)b, lane);
    const unsigned hi = (unsigned)__builtin_amdgcn_readlane((int)(unsigned)(b >> 32), lane);
    return __longlong_as_double((long long)(((unsigned long long)hi << 32) | lo));
}
__device__ __forceinline__ float res_lane(float v, int lane) {
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), lane));
}
// lane 7 (15) of a row: sum of its lanes 0..7 (8..15)
template <typename T>
__device__ __forceinline__ T res_row8(T v) {
    v += res_dpp<0x111, 0xf>(v);   // row_shr:1
    v += res_dpp<0x112, 0xf>(v);   // row_shr:2
    v += res_dpp<0x114, 0xf>(v);   // row_shr:4
    return v;
}
// Sum over the wave, uniform, in a fixed order: shifts within rows of 16
// lanes, then the row sums (six DPP steps instead of six trips through the
// LDS crossbar: about 1 us less per iteration of a one-workgroup CG solve).
template <typename T>
__device__ __forceinline__ T res_wave(T v) {
    v = res_row8(v);
    v += res_dpp<0x118, 0xf>(v);   // row_shr:8
    v += res_dpp<0x142, 0xa>(v);   // row_bcast:15 into rows 1, 3
    v += res_dpp<0x143, 0xc>(v);   // row_bcast:31 into rows 2, 3
    return res_lane(v, 63);
}

}  // namespace mtl4g
