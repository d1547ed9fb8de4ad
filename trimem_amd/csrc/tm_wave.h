// tm_wave.h -- sums over groups of lanes of a wave with DPP lane moves.
#pragma once

#include <hip/hip_runtime.h>

namespace tmh {

// Sums over the 8 lanes of a group with DPP lane moves (no LDS traffic):
// xor 1 and xor 2 within quads, then each lane i of the group pairs with lane
// 7 - i (row_half_mirror), which joins the two quads.  Every lane ends with
// the same bits (the last step adds the same two quad sums, a + b == b + a).
constexpr int kDppXor1 = 0xB1;        // quad_perm [1,0,3,2]
constexpr int kDppXor2 = 0x4E;        // quad_perm [2,3,0,1]
constexpr int kDppHalfMirror = 0x141; // row_half_mirror
template <int CTRL>
__device__ __forceinline__ int dpp_i(int v)
{
    return __builtin_amdgcn_update_dpp(0, v, CTRL, 0xF, 0xF, false);
}
template <int CTRL>
__device__ __forceinline__ double dpp_d(double v)
{
    int lo = __double2loint(v), hi = __double2hiint(v);
    return __hiloint2double(dpp_i<CTRL>(hi), dpp_i<CTRL>(lo));
}
__device__ __forceinline__ double group_sum(double x)
{
    x += dpp_d<kDppXor1>(x);
    x += dpp_d<kDppXor2>(x);
    x += dpp_d<kDppHalfMirror>(x);
    return x;
}
__device__ __forceinline__ int group_sum(int x)
{
    x += dpp_i<kDppXor1>(x);
    x += dpp_i<kDppXor2>(x);
    x += dpp_i<kDppHalfMirror>(x);
    return x;
}
// The 16 lanes of a row: group_sum, then lane i with lane 15 - i (row_mirror).
constexpr int kDppMirror = 0x140;
__device__ __forceinline__ double row_sum(double x)
{
    x = group_sum(x);
    return x + dpp_d<kDppMirror>(x);
}

}    // namespace tmh
