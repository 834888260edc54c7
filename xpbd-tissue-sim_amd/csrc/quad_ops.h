// Device helpers shared by the kernel files: the XCD-contiguous workgroup
// mapping and sums over the four lanes of a DPP quad.
#pragma once
#include <hip/hip_runtime.h>

namespace xpbd {

// Workgroups are dispatched round-robin over the 8 XCDs (workgroup b runs on
// XCD b % 8), and each XCD has its own L2.  With remap set, workgroup b takes
// the work item that gives every XCD one contiguous eighth of the G items:
// neighbouring clusters or patches (adjacent in solver order) then share an L2,
// and since every colour's clusters follow the same spatial order, a vertex
// written in one colour launch is read in the next by the same XCD.
constexpr int kXcds = 8;
__device__ __forceinline__ int xcd_item(int b, int G, bool remap)
{
    if (!remap) return b;
    const int q = G / kXcds, r = G % kXcds, x = b % kXcds;
    return x * q + min(x, r) + b / kXcds;
}

__device__ __forceinline__ float dpp_xor1(float x)
{
    return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(x), 0xB1, 0xF, 0xF, true));
}
__device__ __forceinline__ float dpp_xor2(float x)
{
    return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(x), 0x4E, 0xF, 0xF, true));
}
// Sum of a * b over the four lanes of a quad, (x + swap1) + swap2, the same
// bits in all four lanes.  The product is rounded in every lane first:
// contracted into an FMA, each lane would add its own unrounded product to its
// partners' rounded ones, and the lanes would no longer hold the same sum.
__device__ __forceinline__ float quad_sum_of_product(float a, float b)
{
#pragma clang fp contract(off)
    const float x = a * b;
    const float y = x + dpp_xor1(x);
    return y + dpp_xor2(y);
}
__device__ __forceinline__ float quad_lane3(float x)
{
    return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(x), 0xFF, 0xF, 0xF, true));
}

}  // namespace xpbd
