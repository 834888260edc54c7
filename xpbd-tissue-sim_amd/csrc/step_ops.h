// Parts of a step's first and last launches, shared by the forms that join them
// with what lies next to them.
#pragma once
#include <hip/hip_runtime.h>

#include "kernels.h"

namespace xpbd {

constexpr int kStepBlock = 256;   // threads of these launches; compaction counts hits of that many faces
constexpr int kStepWaves = kStepBlock / 64;

// The inertial move of vertex v (with dz1 the first-order one).
__device__ __forceinline__ float4 predicted(const Prediction& P, int v)
{
    if (P.dz1) return make_float4(0.f, 0.f, P.dz1[v], 0.f);
    const float4 u = P.vel[v];
    return make_float4(P.dt * u.x, P.dt * u.y, P.dt * u.z + P.dz, 0.f);
}

// Hits of a workgroup's faces before this thread's, and in hits of all of them.
__device__ __forceinline__ int hits_before(bool hit, int* ws, int& hits)
{
    const unsigned long long m = __ballot(hit);
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    if (lane == 0) ws[wv] = __popcll(m);
    __syncthreads();
    int before = __popcll(m & ((1ull << lane) - 1ull));
    hits = 0;
#pragma unroll
    for (int w = 0; w < kStepWaves; w++) {
        if (w < wv) before += ws[w];
        hits += ws[w];
    }
    return before;
}

// Ordered compaction of the hit flags, from the hits of each 256 faces, by block b
// of nb: cpos[j] = number of hits before face slot j, cpos[nf] = total,
// clist[cpos[j]] = j for every hit (face order preserved).  Every workgroup adds
// up the counts before its own, some loads a thread (a million faces: 16),
// instead of a launch of its own for that.  ws: 2 kStepWaves ints of LDS.
__device__ __forceinline__ void scatter_hits(const HitLists& H, int b, int nb, int* ws)
{
    const int j = b * kStepBlock + (int)threadIdx.x;
    int* const wb = ws + kStepWaves;
    int sum = 0;
    for (int k = threadIdx.x; k < b; k += kStepBlock) sum += H.bsum[k];
    const bool f = j < H.nf && H.flag[j] != 0;
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) sum += __shfl_xor(sum, o);
    if ((threadIdx.x & 63) == 0) wb[threadIdx.x >> 6] = sum;
    int hits;
    int p = hits_before(f, ws, hits), base = 0;
#pragma unroll
    for (int w = 0; w < kStepWaves; w++) base += wb[w];
    p += base;
    if (j < H.nf) {
        H.cpos[j] = p;
        if (f) H.clist[p] = j;
    }
    if (b == nb - 1 && threadIdx.x == 0) H.cpos[H.nf] = base + hits;
}

}  // namespace xpbd
