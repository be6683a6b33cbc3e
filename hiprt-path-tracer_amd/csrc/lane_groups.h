// lane_groups.h -- a wave as eight groups of eight lanes.
#pragma once

#include <hip/hip_runtime.h>

namespace mipt {

constexpr int GROUP = 8;

// Value of the lane whose index in the group of eight is lane ^ X.
template <int X> __device__ __forceinline__ uint32_t group_xor(uint32_t v)
{
    constexpr int QUAD = X & 4 ? 3 - (X & 3) : X; // half-row mirror is ^ 7
    int r = (int)v;
    if (X & 4)
        r = __builtin_amdgcn_mov_dpp(r, 0x141, 0xf, 0xf, true); // row_half_mirror
    if (QUAD == 1)
        r = __builtin_amdgcn_mov_dpp(r, 0xb1, 0xf, 0xf, true); // quad_perm 1 0 3 2
    else if (QUAD == 2)
        r = __builtin_amdgcn_mov_dpp(r, 0x4e, 0xf, 0xf, true); // quad_perm 2 3 0 1
    else if (QUAD == 3)
        r = __builtin_amdgcn_mov_dpp(r, 0x1b, 0xf, 0xf, true); // quad_perm 3 2 1 0
    return (uint32_t)r;
}

__device__ __forceinline__ uint32_t group_min(uint32_t v)
{
    v = min(v, group_xor<1>(v));
    v = min(v, group_xor<2>(v));
    return min(v, group_xor<7>(v));
}

// Lanes of the group (bit c for lane c) that vote yes.
__device__ __forceinline__ uint32_t group_ballot(bool yes, uint32_t group_shift)
{
    return (uint32_t)(__ballot(yes) >> group_shift) & 0xffu;
}

__device__ __forceinline__ uint32_t group_max(uint32_t v)
{
    v = max(v, group_xor<1>(v));
    v = max(v, group_xor<2>(v));
    return max(v, group_xor<7>(v));
}

__device__ __forceinline__ uint32_t group_or(uint32_t v)
{
    v |= group_xor<1>(v);
    v |= group_xor<2>(v);
    return v | group_xor<7>(v);
}

template <int X> __device__ __forceinline__ float group_xor_f(float v)
{
    return __uint_as_float(group_xor<X>(__float_as_uint(v)));
}

__device__ __forceinline__ float group_min_f(float v)
{
    v = fminf(v, group_xor_f<1>(v));
    v = fminf(v, group_xor_f<2>(v));
    return fminf(v, group_xor_f<7>(v));
}

__device__ __forceinline__ float group_max_f(float v)
{
    v = fmaxf(v, group_xor_f<1>(v));
    v = fmaxf(v, group_xor_f<2>(v));
    return fmaxf(v, group_xor_f<7>(v));
}

} // namespace mipt
