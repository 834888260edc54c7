// Launch wrappers of the vertex-tile Jacobi iteration (jacobi_tile_kernels.hip).
#pragma once
#include <hip/hip_runtime.h>

#include "kernels.h"

namespace xpbd {

// Device views of a JacobiTiles and of its element data.
struct JacobiTileArgs {
    const int* head;          // JacobiTiles::kHead ints a tile
    const uint4* local;       // per tile element: vertices, correction slots, 16 bits each
    const float4* stream;     // three planes of n: Q's nine, alpha tilde D and H, gamma
    const int* home;          // per tile element
    const int4* face;         // per tile face
    const int2* group;
    const uint4* sums;        // per slot, two each
    const int2* out;
    float2* lam;              // per tile element
    float2* dlam;             // solver order
    const float4* din;        // in-step motion by slot
    float4* dout;
    const float4* base;       // base displacement, inverse mass by slot
    const int* vert;          // slot -> vertex, for contacts
    int n;                    // tile elements in all
    int verts, slots;         // room in LDS
    int niter, ntiles, xcd;
    int lam_zero;             // the first iteration's multipliers are zero
    int import;               // they are kept's
    int lam_out;              // the last iteration also writes dlam
    // contacts
    int late;                 // added after all elements
    const int* flag;
    const double *rest, *cp, *cn, *cb;
    const float4* lo;
    double* clam;
    const float2* kept;       // solver order, what an import reads: not dlam where this launch writes that and tiles
                              // share elements
};

size_t jacobi_tile_smem(int verts, int slots);
// once, outside any capture: lets the kernels use all of a workgroup's LDS
hipError_t jacobi_tile_prepare();
hipError_t launch_jacobi_tile(hipStream_t s, const JacobiTileArgs& A, int threads, bool con);
hipError_t launch_jacobi_tile_fill(hipStream_t s, const TetArrays& ta, const int* home, int n, float4* stream);

}  // namespace xpbd
