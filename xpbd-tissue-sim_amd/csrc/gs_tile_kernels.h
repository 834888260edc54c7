// Launch wrappers of the fused-colour Gauss-Seidel kernels (gs_tile_kernels.hip).
#pragma once
#include <hip/hip_runtime.h>
#include <cstdint>

#include "kernels.h"

namespace xpbd {

constexpr size_t kGsTileLds = 160 * 1024;   // LDS of a workgroup, gfx950

constexpr int kLaneRow = 224;   // float4s of 64 elements' data with one lane a cluster

// Which tile kernel: lanes per cluster (4 or 1), element rows of a block at
// most (6 or 8), and whether every block has that many (always so with one lane).
struct GsTileShape {
    int lanes = 4, rows = 6;
    bool full = false;
    int cap = 0;   // one lane a cluster: slots that the LDS layout has room for (gs_tile_cap)
};

// Device views of a GsTileGroup and of its element data.
struct GsTileArgs {
    const int2* tile;        // per tile: barriers an iteration, entries of out
    const int2* wave;        // per tile and wave: blocks, barriers before the first
    const int* list;         // per tile, wave and block: element rows | barriers until the wave's next << 4
    const int2* out;         // per tile: slot of the tile, slot of dout
    const int* home;         // one lane a cluster: per block and lane 2 * first solver position + whether it writes dlam
    const float4* stream;    // four lanes a cluster, 64 per row: lane j of a quad (Q's row j, then alpha tilde D / H /
                             // gamma); a block's first row: eight 16-bit slots a lane.
                             // One lane a cluster, kLaneRow per row: see k_gs_tile_lane
    float2* lam;             // 16 (64) per row; with four lanes a block's first row: as home
    float2* dlam;            // solver order
    const float4* din;       // in-step motion, by slot of this group
    float4* dout;            // by slot of the next
    const float4* base;      // base displacement, inverse mass, by slot
    int waves, slots, rows, blocks, outs;   // strides: see GsTileGroup
    int niter, nt;
    int lam_zero;            // the first iteration's multipliers are zero
    int lam_out;             // the last iteration also writes dlam
    const float2* kept;      // solver order, what an import reads: not dlam where this launch writes that and tiles
                             // share clusters.  Last: between the others it moved the kernel's loads of them, beam
                             // 200x20x20 474 -> 477 us a step
};

struct GsTileFill {
    TetArrays ta;
    const int* cstart;
    const uint32_t* tloc;
    const int* list;
    const int* row;
    const int* clu;
    const uint8_t* own;
    const uint16_t* vert;
    float4* stream;
    float2* lam;
    int* home;               // one lane a cluster
    int nblocks, slots;
};

size_t gs_tile_smem(int slots, const GsTileShape& S);
int gs_tile_cap(int slots);   // 0: too many for one lane a cluster
// once per shape, outside any capture: lets the kernel use kGsTileLds bytes of LDS
hipError_t gs_tile_prepare(const GsTileShape& S);
// import: the first iteration's multipliers come from kept
hipError_t launch_gs_tile(hipStream_t s, const GsTileArgs& A, const GsTileShape& S, int ntiles, int threads, size_t smem,
                          bool import);
hipError_t launch_gs_tile_fill(hipStream_t s, const GsTileFill& A, const GsTileShape& S);
// bases of the vertex records into n slots, in-step motions into the first nd; motions back
hipError_t launch_gs_tile_load(hipStream_t s, const float4* pos, const int* slot_vert, int n, int nd, float4* d,
                               float4* base, const Prediction* predict = nullptr, const HitLists* hits = nullptr);
hipError_t launch_gs_tile_store(hipStream_t s, float4* pos, const int* owner, int nv, const float4* d);

}  // namespace xpbd
