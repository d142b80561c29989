// lanes.h -- values of other lanes of a wavefront (gfx950, 64 lanes).
#pragma once

#include <hip/hip_runtime.h>

namespace fdtd {

// lane l receives lane l-1's (lane l+1's) value; lane 0 (63) receives 0
__device__ __forceinline__ int dpp_left(int v)
{
    return __builtin_amdgcn_update_dpp(0, v, 0x138 /* wave_shr:1 */, 0xf, 0xf, false);
}
__device__ __forceinline__ int dpp_right(int v)
{
    return __builtin_amdgcn_update_dpp(0, v, 0x130 /* wave_shl:1 */, 0xf, 0xf, false);
}
struct Int2 { int lo, hi; };
__device__ __forceinline__ float lane_left(float v)
{
    return __builtin_bit_cast(float, dpp_left(__builtin_bit_cast(int, v)));
}
__device__ __forceinline__ float lane_right(float v)
{
    return __builtin_bit_cast(float, dpp_right(__builtin_bit_cast(int, v)));
}
__device__ __forceinline__ double lane_left(double v)
{
    const Int2 q = __builtin_bit_cast(Int2, v);
    return __builtin_bit_cast(double, Int2{dpp_left(q.lo), dpp_left(q.hi)});
}
__device__ __forceinline__ double lane_right(double v)
{
    const Int2 q = __builtin_bit_cast(Int2, v);
    return __builtin_bit_cast(double, Int2{dpp_right(q.lo), dpp_right(q.hi)});
}
// lane `lane`'s value, in every lane
__device__ __forceinline__ float lane_get(float v, int lane)
{
    return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), lane));
}
__device__ __forceinline__ double lane_get(double v, int lane)
{
    const Int2 q = __builtin_bit_cast(Int2, v);
    return __builtin_bit_cast(double, Int2{__builtin_amdgcn_readlane(q.lo, lane),
                                           __builtin_amdgcn_readlane(q.hi, lane)});
}
// the value of the lane that each lane names (from: 4 times its number)
__device__ __forceinline__ float lane_pick(float v, int from)
{
    return __builtin_bit_cast(float, __builtin_amdgcn_ds_bpermute(from, __builtin_bit_cast(int, v)));
}
__device__ __forceinline__ double lane_pick(double v, int from)
{
    const Int2 q = __builtin_bit_cast(Int2, v);
    return __builtin_bit_cast(double, Int2{__builtin_amdgcn_ds_bpermute(from, q.lo),
                                           __builtin_amdgcn_ds_bpermute(from, q.hi)});
}

}  // namespace fdtd
