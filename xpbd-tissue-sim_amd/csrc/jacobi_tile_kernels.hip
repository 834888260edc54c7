// Vertex-tile Jacobi iteration: one launch an iteration, a workgroup a tile (see
// jacobi_tiles.h).
#include "jacobi_tile_kernels.h"

#include "contact_ops.h"
#include "jacobi_tiles.h"
#include "quad_ops.h"
#include "xpbd_math.h"

namespace xpbd {
namespace {

constexpr int kTileThreads = 1024;

struct TileTet {
    uint4 idx;
    float q[9], atD, atH, gm;
    float2 l;
};

// an own vertex's JacobiTiles::sums and its group
struct SumOf {
    uint4 m, c;
    int2 g;
};

constexpr int kAhead = 8;   // corrections read together

// The elements' corrections of one component of a vertex, partial sums by patch; CON:
// with the contacts' partial sums c, in their order.  What is read past the last
// correction follows the last end of a partial sum, so it goes nowhere.
template <bool CON>
__device__ __forceinline__ float sum_elements(const SumOf& q, const float* r, const float* c)
{
    const int nt = q.c.x & 0xffffu;
    float total = 0.f, s = 0.f;
    int nc = 0;
    uint32_t end = q.m.x, con = q.m.z;
    for (int e0 = 0; e0 < nt; e0 += kAhead) {
        if (e0 == 32) {
            end = q.m.y;
            con = q.m.w;
        }
        float v[kAhead];
#pragma unroll
        for (int u = 0; u < kAhead; u++) v[u] = r[q.g.x + 64 * (e0 + u)];
#pragma unroll
        for (int u = 0; u < kAhead; u++) {
            s += v[u];
            if (CON && (con >> u & 1u)) s += c[64 * nc++];
            const bool ends = end >> u & 1u;
            total = ends ? total + s : total;
            s = ends ? 0.f : s;
        }
        end >>= kAhead;
        con >>= kAhead;
    }
    return total;
}

// The same with contacts: their partial sums go to the front of their slots.  Sums of
// nothing but zeros (no contact is active) need not be added.
__device__ __forceinline__ float sum_contacts(const SumOf& q, float* r, int late)
{
    const int nf = q.c.x >> 16;
    float* const c = r + q.g.y;
    float t = 0.f, all = 0.f;
    int nc = 0;
    for (int f0 = 0; f0 < nf; f0 += kAhead) {
        float v[kAhead];
#pragma unroll
        for (int u = 0; u < kAhead; u++) v[u] = c[64 * min(f0 + u, nf - 1)];
#pragma unroll
        for (int u = 0; u < kAhead; u++)
            if (f0 + u < nf) {
                t += v[u];
                if (q.c.y >> (f0 + u) & 1u) {
                    c[64 * nc++] = t;
                    all = t != 0.f ? t : all;
                    t = 0.f;
                }
            }
    }
    if (!__any(all != 0.f)) return sum_elements<false>(q, r, nullptr);
    if (!late) return sum_elements<true>(q, r, c);
    const float total = sum_elements<false>(q, r, nullptr);
    return nf > 0 ? total + c[0] : total;
}

__device__ __forceinline__ void load_tile_tet(const JacobiTileArgs& A, int i, bool first, TileTet& t)
{
    t.idx = A.local[i];
    const float4 a = A.stream[i], b = A.stream[(size_t)A.n + i], c = A.stream[2 * (size_t)A.n + i];
    t.q[0] = a.x, t.q[1] = a.y, t.q[2] = a.z, t.q[3] = a.w;
    t.q[4] = b.x, t.q[5] = b.y, t.q[6] = b.z, t.q[7] = b.w;
    t.q[8] = c.x, t.atD = c.y, t.atH = c.z, t.gm = c.w;
    t.l = first && A.lam_zero ? make_float2(0.f, 0.f) : first && A.import ? A.kept[A.home[i] >> 1] : A.lam[i];
}

// An element's projection from the tile's motions; corrections of own vertices to their slots.
__device__ __forceinline__ void project_tile_tet(TileTet& t, const float4* lb, const float4* ld, float* red, int slots)
{
    const int v[4] = { (int)(t.idx.x & 0xffffu), (int)(t.idx.x >> 16), (int)(t.idx.y & 0xffffu), (int)(t.idx.y >> 16) };
    const int s[4] = { (int)(t.idx.z & 0xffffu), (int)(t.idx.z >> 16), (int)(t.idx.w & 0xffffu), (int)(t.idx.w >> 16) };
    float bb[12], dd[12], w[4], l[2] = { t.l.x, t.l.y }, dx[12];
#pragma unroll
    for (int j = 0; j < 4; j++) {
        const float4 b = lb[v[j]], d = ld[v[j]];
        bb[3 * j] = b.x, bb[3 * j + 1] = b.y, bb[3 * j + 2] = b.z;
        dd[3 * j] = d.x, dd[3 * j + 1] = d.y, dd[3 * j + 2] = d.z;
        w[j] = b.w;
    }
    project_tet_split<float, true>(bb, dd, w, t.q, t.atD, t.atH, t.gm, l, dx);
    t.l = make_float2(l[0], l[1]);
#pragma unroll
    for (int j = 0; j < 4; j++)
        if (s[j] != 0xffff)
#pragma unroll
            for (int k = 0; k < 3; k++) red[k * slots + s[j]] = dx[3 * j + k];
}

// The contact of a tile's face from the same motions, in FP64; corrections (zeros
// without a contact) to the face slots of own vertices.
__device__ __forceinline__ void project_tile_face(const JacobiTileArgs& A, int4 F, int v0, bool first, const float4* lb,
                                                  const float4* ld, float* red)
{
    const int j = F.x >> 1;
    const int v[3] = { F.y & 0xffff, (int)((unsigned)F.y >> 16), F.z & 0xffff };
    const int s[3] = { (int)((unsigned)F.z >> 16), F.w & 0xffff, (int)((unsigned)F.w >> 16) };
    double dx[9];
    bool act = false;
    if (A.flag[j]) {
        double x[3][3];
        float w[3];
#pragma unroll
        for (int m = 0; m < 3; m++) {
            const int g = A.vert[v0 + v[m]];
            const float4 b = lb[v[m]], d = ld[v[m]], lo = A.lo[g];
            x[m][0] = A.rest[3 * (size_t)g] + (((double)b.x + (double)lo.x) + (double)d.x);
            x[m][1] = A.rest[3 * (size_t)g + 1] + (((double)b.y + (double)lo.y) + (double)d.y);
            x[m][2] = A.rest[3 * (size_t)g + 2] + (((double)b.z + (double)lo.z) + (double)d.z);
            w[m] = b.w;
        }
        const double* xs[3] = { x[0], x[1], x[2] };
        double lam = 0.0;
        if ((F.x & 1) && !first) lam = A.clam[j];
        act = contact_dx(xs, w, A.cp + 3 * (size_t)j, A.cn + 3 * (size_t)j, A.cb + 3 * (size_t)j, &lam, dx);
        if (F.x & 1) A.clam[j] = lam;
    }
#pragma unroll
    for (int m = 0; m < 3; m++)
        if (s[m] != 0xffff)
#pragma unroll
            for (int k = 0; k < 3; k++) red[k * A.slots + s[m]] = act ? (float)dx[3 * m + k] : 0.f;
}

// One iteration of a tile (all of them where tiles are closed): motions to LDS,
// every element projected by a thread, its corrections to one LDS slot for each
// vertex the tile owns, then a thread for each component of an own vertex sums its
// slots (side by side for the 64 of a group: no bank conflicts).  12^3 cells: 5 us,
// the chain of launch, loads, one projection and one sum; beam 200x20x20: 17 us,
// three elements a thread at 4 waves a SIMD (116 registers), the projection's
// instructions.  Tried there: the next element's data in flight while one is
// projected (copies of 20 registers: 184 us a step against 171), 512 threads and
// tiles of half the size (173), spare slots instead of branches for other tiles'
// vertices (no gain, more LDS writes).  The sums keep the patch launches' grouping,
// and so their bits, for 0.2 us an iteration: Jacobi under contact amplifies rounding
// tenfold in ten steps.
template <bool CON>
__global__ __launch_bounds__(kTileThreads) void k_jacobi_tile(JacobiTileArgs A)
{
    extern __shared__ float4 lds[];
    float4 *const lb = lds, *const ld = lds + A.verts;
    float* const red = reinterpret_cast<float*>(lds + 2 * A.verts);
    const int tid = threadIdx.x, nthreads = blockDim.x;
    const int* h = A.head + JacobiTiles::kHead * xcd_item(blockIdx.x, gridDim.x, A.xcd != 0);
    const int v0 = h[JacobiTiles::V0], nv = h[JacobiTiles::NV], own = h[JacobiTiles::OWN], t0 = h[JacobiTiles::T0],
              nt = h[JacobiTiles::NT], f0 = h[JacobiTiles::F0], nf = h[JacobiTiles::NF], o0 = h[JacobiTiles::O0],
              no = h[JacobiTiles::NO], g0 = h[JacobiTiles::G0];
    TileTet t;   // a thread's first element; its only one stays with it
    if (tid < nt) load_tile_tet(A, t0 + tid, true, t);
    for (int i = tid; i < nv; i += nthreads) {
        lb[i] = A.base[v0 + i];
        ld[i] = A.din[v0 + i];
    }
    // how a thread's first sum is grouped
    const int width = (own + 63) & ~63;
    auto sum_of = [&](int o) {
        return SumOf{ A.sums[2 * (size_t)(v0 + o)], A.sums[2 * (size_t)(v0 + o) + 1], A.group[g0 + (o >> 6)] };
    };
    SumOf mine{};
    {
        const int o = tid - ((tid >= width) + (tid >= 2 * width)) * width;
        if (o < own) mine = sum_of(o);
    }
    __syncthreads();
    for (int it = 0; it < A.niter; it++) {
        const bool first = it == 0, last = it == A.niter - 1;
        for (int i = tid; i < nt; i += nthreads) {
            if (i == tid) {
                project_tile_tet(t, lb, ld, red, A.slots);
                if (last) A.lam[t0 + i] = t.l;
                if (last && A.lam_out) {
                    const int home = A.home[t0 + i];
                    if (home & 1) A.dlam[home >> 1] = t.l;
                }
                continue;
            }
            TileTet u;
            load_tile_tet(A, t0 + i, first, u);
            project_tile_tet(u, lb, ld, red, A.slots);
            A.lam[t0 + i] = u.l;
            if (last && A.lam_out) {
                const int home = A.home[t0 + i];
                if (home & 1) A.dlam[home >> 1] = u.l;
            }
        }
        if (CON)
            for (int i = tid; i < nf; i += nthreads)
                project_tile_face(A, A.face[f0 + i], v0, first && A.lam_zero, lb, ld, red);
        __syncthreads();
        // a thread sums one component of one vertex, grouped as the patch launches do
        for (int x = tid; x < 3 * width; x += nthreads) {
            const int k = (x >= width) + (x >= 2 * width), o = x - k * width;
            if (o >= own) continue;
            const SumOf q = x == tid ? mine : sum_of(o);
            float total;
            if constexpr (CON) total = sum_contacts(q, red + k * A.slots + (o & 63), A.late);
            else total = sum_elements<false>(q, red + k * A.slots + (o & 63), nullptr);
            reinterpret_cast<float*>(ld)[4 * o + k] += total;
        }
        __syncthreads();
    }
    for (int i = tid; i < no; i += nthreads) {
        const int2 o = A.out[o0 + i];
        A.dout[o.y] = ld[o.x];
    }
}

__global__ __launch_bounds__(256) void k_jacobi_tile_fill(TetArrays ta, const int* __restrict__ home, int n,
                                                         float4* __restrict__ stream)
{
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i >= n) return;
    const int e = home[i] >> 1;
    float q[9];
#pragma unroll
    for (int k = 0; k < 9; k++) q[k] = ta.Q[(size_t)k * ta.qstride + e];
    const float2 at = ta.at[e];
    stream[i] = make_float4(q[0], q[1], q[2], q[3]);
    stream[(size_t)n + i] = make_float4(q[4], q[5], q[6], q[7]);
    stream[2 * (size_t)n + i] = make_float4(q[8], at.x, at.y, ta.gamma[e]);
}

}  // namespace

// with the room that a vertex's last reads may run into
size_t jacobi_tile_smem(int verts, int slots) { return 32 * (size_t)verts + 12 * (size_t)slots + 4 * 64 * kAhead; }

hipError_t jacobi_tile_prepare()
{
    hipError_t e = hipSuccess;
    for (const void* k : { reinterpret_cast<const void*>(k_jacobi_tile<false>), reinterpret_cast<const void*>(k_jacobi_tile<true>) })
        if (e == hipSuccess) e = hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
    return e;
}

hipError_t launch_jacobi_tile(hipStream_t s, const JacobiTileArgs& A, int threads, bool con)
{
    if (A.ntiles <= 0 || A.niter <= 0) return hipSuccess;
    if (threads < 64 || threads > kTileThreads || threads % 64) return hipErrorInvalidValue;
    const size_t smem = jacobi_tile_smem(A.verts, A.slots);
    if (con) hipLaunchKernelGGL(k_jacobi_tile<true>, dim3(A.ntiles), dim3(threads), smem, s, A);
    else hipLaunchKernelGGL(k_jacobi_tile<false>, dim3(A.ntiles), dim3(threads), smem, s, A);
    return hipGetLastError();
}

hipError_t launch_jacobi_tile_fill(hipStream_t s, const TetArrays& ta, const int* home, int n, float4* stream)
{
    if (n <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_jacobi_tile_fill, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, ta, home, n, stream);
    return hipGetLastError();
}

}  // namespace xpbd
