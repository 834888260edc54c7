// Fused-colour Gauss-Seidel: one launch projects a group of consecutive
// colours (gs_tiles.h), a workgroup per tile.
//
// A colour launch of the quad cluster kernel on a mesh of 10^5..10^6 elements
// holds about one wave per SIMD and spends more on its launch, on the two
// dependent loads before the first projection and on re-staging every vertex
// than on the projections.  Here a workgroup stages its tile's vertices in LDS
// once, runs the group's colours with a workgroup barrier between them, and
// writes back the vertices it owns.  Element data are kept per tile in the
// order and lane in which they are used: one 16-byte load a lane for an
// element, issued while the wave's previous block of that slot is projected,
// so no load of theirs is on the dependent chain after a launch's first block.
#include <hip/hip_runtime.h>

#include "gs_tile_kernels.h"
#include "quad_ops.h"
#include "step_ops.h"
#include "xpbd_math.h"

namespace xpbd {

namespace {

// A workgroup barrier for what the waves share, which is LDS: global loads in
// flight (the next block's element data) are not waited for.
__device__ __forceinline__ void lds_barrier()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

template <int LANE>
__device__ __forceinline__ float quad_from(float x)
{
    return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(x), LANE * 0x55, 0xF, 0xF, true));
}

// One element of a quad: lane j holds its vertex's base and inverse mass b and
// in-step motion d, and q = (row j of Q; alpha tilde D, alpha tilde H, gamma in
// lanes 0..2).  The same operations, in the same order, as the quad cluster
// kernel's step, so the same bits.  Updates d and lam.
__device__ __forceinline__ void project_quad(const float4 q, const float4 b, float (&d)[3], float2& lam)
{
    const float qj[3] = { q.x, q.y, q.z };
    const float atD = quad_from<0>(q.w), atH = quad_from<1>(q.w), gamma = quad_from<2>(q.w);
    const float bb[3] = { b.x, b.y, b.z };
    const float w = b.w;
    float D[3];
#pragma unroll
    for (int k = 0; k < 3; k++) D[k] = (bb[k] - quad_lane3(bb[k])) + (d[k] - quad_lane3(d[k]));
    float F[9];
#pragma unroll
    for (int c = 0; c < 3; c++)
#pragma unroll
        for (int r = 0; r < 3; r++) {
            const float sum = quad_sum_of_product(D[r], qj[c]);
            F[3 * c + r] = r == c ? sum + 1.f : sum;
        }
    float ss = 0.f;
#pragma unroll
    for (int i = 0; i < 9; i++) ss += F[i] * F[i];
    const float CD = xsqrt<float>(ss);
    float Fc[9];
    Fc[0] = F[4] * F[8] - F[5] * F[7];
    Fc[1] = F[5] * F[6] - F[3] * F[8];
    Fc[2] = F[3] * F[7] - F[4] * F[6];
    Fc[3] = F[7] * F[2] - F[8] * F[1];
    Fc[4] = F[8] * F[0] - F[6] * F[2];
    Fc[5] = F[6] * F[1] - F[7] * F[0];
    Fc[6] = F[1] * F[5] - F[2] * F[4];
    Fc[7] = F[2] * F[3] - F[0] * F[5];
    Fc[8] = F[0] * F[4] - F[1] * F[3];
    const float J = F[0] * Fc[0] + F[1] * Fc[1] + F[2] * Fc[2];
    const float a = J - 1.f;
    const float ch_log = -gamma + xlog<float>(J);
    const float ch_series = -gamma + a - a * a * 0.5f + a * a * a * (1.f / 3.f);
    const float CH = J >= 1.f ? ch_log : ch_series;
    const float inv_C = xrcp<float>(CD);
    const float fac = (J >= 1.f) ? xrcp<float>(J) : 1.f - a + a * a;
    float gD[3], gH[3];
#pragma unroll
    for (int r = 0; r < 3; r++) {
        gD[r] = inv_C * (F[r] * qj[0] + F[3 + r] * qj[1] + F[6 + r] * qj[2]);
        gH[r] = fac * (Fc[r] * qj[0] + Fc[3 + r] * qj[1] + Fc[6 + r] * qj[2]);
    }
    const float s00 = quad_sum_of_product(w, gD[0] * gD[0] + gD[1] * gD[1] + gD[2] * gD[2]);
    const float s01 = quad_sum_of_product(w, gD[0] * gH[0] + gD[1] * gH[1] + gD[2] * gH[2]);
    const float s11 = quad_sum_of_product(w, gH[0] * gH[0] + gH[1] * gH[1] + gH[2] * gH[2]);
    const float A00 = atD + s00, A11 = atH + s11, A01 = s01;
    const float b0 = -CD - atD * lam.x;
    const float b1 = -CH - atH * lam.y;
    // SPD in exact arithmetic; a non-positive FP32 determinant (slivers) skips
    // the projection, as in project_tet_F
    const float det = A00 * A11 - A01 * A01;
    const float inv_det = det > 0.f ? xrcp<float>(det) : 0.f;
    const float d0 = (b0 * A11 - b1 * A01) * inv_det;
    const float d1 = (b1 * A00 - b0 * A01) * inv_det;
    lam.x += d0;
    lam.y += d1;
#pragma unroll
    for (int k = 0; k < 3; k++) d[k] = d[k] + w * (gD[k] * d0 + gH[k] * d1);
}

// Both tile kernels.  Everything a wave needs first lies where (tile, wave,
// thread) says: its slots' motions and bases, its first rows, its block list.
// So all of it is asked for at once, and no address waits for a load.
// slots a thread stages at a time (KS below): fewer where registers are short
constexpr int kStageQuad = 3, kStageLane = 5;
constexpr int kOut = 4;     // results whose places a thread knows before it computes

// The tile's slots: the first KS of a thread are loaded, then stored (with
// other loads issued between), the others loaded and stored in turn.
// store(slot, base, motion).
template <int KS>
struct TileStage {
    float4 d[KS], b[KS];
};
template <int KS>
__device__ __forceinline__ void tile_load(const GsTileArgs& A, int t, int i0, TileStage<KS>& g)
{
    const float4* din = A.din + (size_t)t * A.slots;
    const float4* base = A.base + (size_t)t * A.slots;
#pragma unroll
    for (int u = 0; u < KS; u++) {
        const int i = min(i0 + u * (int)blockDim.x, A.slots - 1);
        g.d[u] = din[i];
        g.b[u] = base[i];
    }
}
template <int KS, typename Store>
__device__ __forceinline__ void tile_stage(const GsTileArgs& A, int t, TileStage<KS>& g, Store store)
{
    for (int i0 = threadIdx.x;;) {
        // past the end the last slot again: the same values to the same place
#pragma unroll
        for (int u = 0; u < KS; u++) store(min(i0 + u * (int)blockDim.x, A.slots - 1), g.b[u], g.d[u]);
        i0 += KS * blockDim.x;
        if (i0 - (int)threadIdx.x >= A.slots) break;   // the same for every thread
        tile_load(A, t, i0, g);
    }
}

// Where the tile's results go: the first kOut of a thread are loaded before it
// computes.
struct TileOut {
    int2 o[kOut];
};
__device__ __forceinline__ TileOut tile_out(const GsTileArgs& A, int t)
{
    TileOut r;
#pragma unroll
    for (int u = 0; u < kOut; u++)
        r.o[u] = A.out[(size_t)t * A.outs + min((int)(threadIdx.x + u * blockDim.x), A.outs - 1)];
    return r;
}
template <typename Read>
__device__ __forceinline__ void tile_write(const GsTileArgs& A, const TileOut& r, int t, int n, Read read)
{
    const int tid = threadIdx.x;
#pragma unroll
    for (int u = 0; u < kOut; u++)
        if (tid + u * (int)blockDim.x < n) A.dout[r.o[u].y] = read(r.o[u].x);
    for (int i = tid + kOut * blockDim.x; i < n; i += blockDim.x) {
        const int2 o = A.out[(size_t)t * A.outs + i];
        A.dout[o.y] = read(o.x);
    }
}

// A wave runs its list of blocks (16 clusters of one colour each).  A list
// entry is the block's element rows | barriers until the wave's next block << 4;
// every wave takes as many barriers an iteration.
// While it projects element row k of a block, a wave loads row k of its next
// block, so the loads have a whole block to arrive; a wave's last block of the
// launch loads its first one again, so that every path issues the same loads
// and the waits count them exactly.
// FULL: every block has MT element rows (each cluster a hexahedral cell).
// IMPORT: the multipliers come from a solver-order array (launches of one iteration).
template <int MT, bool FULL, bool IMPORT>
__global__ __launch_bounds__(1024) void k_gs_tile(GsTileArgs A)
{
    extern __shared__ float4 lds[];
    float4* const sb = lds;                                    // base, inverse mass
    float* const sd = reinterpret_cast<float*>(lds + A.slots);  // in-step motion, 3 floats a slot
    const int lane = threadIdx.x & 63, j = lane & 3, quad = lane >> 2;
    const int t = xcd_item(blockIdx.x, gridDim.x, true);
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const size_t tw = (size_t)t * A.waves + min(wave, A.waves - 1);   // waves past the last only stage
    const int2 tile = A.tile[t], head = A.wave[tw];
    const int* list = A.list + tw * A.blocks;
    int cur = list[0], nxt = list[min(1, A.blocks - 1)];
    TileStage<kStageQuad> g;
    tile_load(A, t, threadIdx.x, g);
    __builtin_amdgcn_sched_barrier(0);   // these return first
    // a block's row 0 holds the vertices' slots (and, in the multiplier array, the
    // solver position), then one row an element
    const float4* const st0 = A.stream + tw * A.rows * 64 + lane;
    float2* const sl0 = A.lam + tw * A.rows * 16 + quad;
    float4 S[MT];
    float2 L[MT];
    uint4 X;
    int H;
    auto load_meta = [&](const float4* st, const float2* sl, uint4& x, int& h) {
        x = *reinterpret_cast<const uint4*>(st);
        h = __float_as_int(sl->x);
    };
    auto load_row = [&](const float4* st, const float2* sl, int k, int rows, bool import, int h) {
        const int r = 1 + (FULL ? k : max(0, min(k, rows - 1)));
        S[k] = st[r * 64];
        L[k] = import ? A.kept[min((h >> 1) + k, A.nt - 1)] : sl[r * 16];
    };
    const int nb = wave < A.waves ? head.x : 0;
    auto first_rows = [&] {
        load_meta(st0, sl0, X, H);
#pragma unroll
        for (int k = 0; k < MT; k++) load_row(st0, sl0, k, cur & 15, IMPORT, H);
    };
    // the rows of the first phase arrive with the slots, those of later phases
    // after them: all workgroups start at once, and what they ask for together
    // is as much as the memory gives in several microseconds
    if (nb > 0 && head.y == 0) first_rows();
    __builtin_amdgcn_sched_barrier(0);
    tile_stage(A, t, g, [&](int i, const float4 b, const float4 d) {
        sb[i] = b;
        sd[3 * i] = d.x;
        sd[3 * i + 1] = d.y;
        sd[3 * i + 2] = d.z;
    });
    lds_barrier();
    if (nb > 0 && head.y > 0) first_rows();
    const TileOut to = tile_out(A, t);
    if (nb == 0) {
        for (int i = A.niter * tile.x; i > 0; i--) lds_barrier();
    } else {
        if (nb == 1) nxt = cur;
        auto slot = [](const uint4& x, int k) {
            const uint32_t w = k < 2 ? x.x : k < 4 ? x.y : k < 6 ? x.z : x.w;
            return (int)((w >> (16 * (k & 1))) & 0xffffu);
        };
        // slot and base of the row to come: they do not wait for the one before it
        // (not where blocks have fewer rows than MT: the next row is not known here)
        int v = slot(X, 0);
        float4 b = sb[v];
        for (int it = 0; it < A.niter; it++) {
            const bool zero = !IMPORT && it == 0 && A.lam_zero;
            const bool last = A.lam_out && it == A.niter - 1;
            for (int i = head.y; i > 0; i--) lds_barrier();
            const float4* st = st0;
            float2* sl = sl0;
            for (int i = 0; i < nb; i++) {
                const int ent = __builtin_amdgcn_readfirstlane(nxt);
                nxt = list[i + 2 < nb ? i + 2 : min(i + 2 - nb, nb - 1)];
                const int cnt = cur & 15, step = FULL ? MT + 1 : cnt + 1;
                const float4* const stn = i + 1 < nb ? st + step * 64 : st0;
                float2* const sln = i + 1 < nb ? sl + step * 16 : sl0;
                uint4 Xn;
                int Hn;
                load_meta(stn, sln, Xn, Hn);
#pragma unroll
                for (int k = 0; k < MT; k++) {
                    if (FULL || k < cnt) {
                        if (!FULL) {
                            v = slot(X, k);
                            b = sb[v];
                        }
                        const int u = v;
                        const float4 bb = b, e = S[k];
                        float d[3] = { sd[3 * u], sd[3 * u + 1], sd[3 * u + 2] };
                        if (FULL) {
                            v = k + 1 < MT ? slot(X, k + 1) : slot(Xn, 0);
                            b = sb[v];
                        }
                        float2 l = L[k];
                        if (zero) l = make_float2(0.f, 0.f);
                        project_quad(e, bb, d, l);
                        sd[3 * u] = d[0];
                        sd[3 * u + 1] = d[1];
                        sd[3 * u + 2] = d[2];
                        // all four lanes hold and store the same value: the load of the
                        // next iteration's copy follows each lane's own store
                        sl[(1 + k) * 16] = l;
                        if (last) {
                            if ((H & 1) && j == 0 && u != A.slots - 1) A.dlam[(H >> 1) + k] = l;
                        }
                        // the next element's reads of other lanes' vertices follow these
                        // writes in program order (LDS operations of one wave complete in order)
                        __builtin_amdgcn_wave_barrier();
                    }
                    load_row(stn, sln, k, ent & 15, IMPORT, Hn);
                }
                for (int n = cur >> 4; n > 0; n--) lds_barrier();
                X = Xn;
                H = Hn;
                cur = ent;
                st = stn;
                sl = sln;
            }
        }
    }
    tile_write(A, to, t, tile.y, [&](int i) { return make_float4(sd[3 * i], sd[3 * i + 1], sd[3 * i + 2], 0.f); });
}

// Lays out a group's element data for k_gs_tile: a thread per (block, quad lane).
__global__ __launch_bounds__(256) void k_gs_tile_fill(GsTileFill A)
{
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i >= A.nblocks * 64) return;
    const int b = i >> 6, lane = i & 63, j = lane & 3, quad = lane >> 2;
    const int rows = A.list[b] & 15;
    if (rows == 0) return;
    const size_t row = (size_t)A.row[b];
    const int c = A.clu[i >> 2];
    const int e0 = c >= 0 ? A.cstart[c] : 0, n = c >= 0 ? A.cstart[c + 1] - e0 : 0;
    uint32_t ix[4];
    for (int k = 0; k < 4; k++) ix[k] = (uint32_t)(A.slots - 1) * 0x10001u;
    for (int k = 0; k < rows; k++) {
        float4 o = make_float4(0.f, 0.f, 0.f, 0.f);
        if (k < n) {
            const int e = e0 + k;
            float q[3];
            for (int cc = 0; cc < 3; cc++) {
                const float q0 = A.ta.Q[(size_t)(3 * cc) * A.ta.qstride + e];
                const float q1 = A.ta.Q[(size_t)(3 * cc + 1) * A.ta.qstride + e];
                const float q2 = A.ta.Q[(size_t)(3 * cc + 2) * A.ta.qstride + e];
                q[cc] = j == 0 ? q0 : j == 1 ? q1 : j == 2 ? q2 : -(q0 + q1 + q2);
            }
            const float2 at = A.ta.at[e];
            o = make_float4(q[0], q[1], q[2], j == 0 ? at.x : j == 1 ? at.y : j == 2 ? A.ta.gamma[e] : 0.f);
            const uint32_t v = A.vert[(size_t)(i >> 2) * 8 + ((A.tloc[e] >> (4 * j)) & 15u)];
            ix[k / 2] = k & 1 ? (ix[k / 2] & 0xffffu) | v << 16 : (ix[k / 2] & 0xffff0000u) | v;
        }
        A.stream[(row + 1 + k) * 64 + lane] = o;
        if (j == 0) A.lam[(row + 1 + k) * 16 + quad] = make_float2(0.f, 0.f);
    }
    *reinterpret_cast<uint4*>(A.stream + row * 64 + lane) = make_uint4(ix[0], ix[1], ix[2], ix[3]);
    if (j == 0) A.lam[row * 16 + quad] = make_float2(__int_as_float(2 * e0 + (A.own[i >> 2] ? 1 : 0)), 0.f);
}

// The sums that project_quad forms over a quad's lanes, in one lane: every product
// rounded, (0 + 1) + (2 + 3).
__device__ __forceinline__ float sum_of_products(const float (&a)[4], const float (&b)[4])
{
#pragma clang fp contract(off)
    const float x0 = a[0] * b[0], x1 = a[1] * b[1], x2 = a[2] * b[2], x3 = a[3] * b[3];
    return (x0 + x1) + (x2 + x3);
}
__device__ __forceinline__ float sum_of_products(float a0, float b0, float a1, float b1, float a2, float b2)
{
#pragma clang fp contract(off)   // the fourth is zero: a position relative to itself
    const float x0 = a0 * b0, x1 = a1 * b1, x2 = a2 * b2;
    return (x0 + x1) + x2;
}

__device__ __forceinline__ float sum3(float a0, float b0, float a1, float b1, float a2, float b2)
{
    return fmaf(a2, b2, fmaf(a0, b0, a1 * b1));
}

// One element in one lane: b its vertices' bases (and inverse masses), d their
// in-step motions, q column-major Q.  The same operations, in the same order, as
// project_quad, so the same bits, with the gradients of all four vertices in turn;
// the FMAs that the compiler makes of its expressions are written out, as it does
// not choose them alike here.  (The 2x2 system's sums by way of M = sum w q q^T need
// 15 % fewer instructions and 24 bytes more an element; but another order of
// operations is another last bit, and where a contact comes or goes by it, another
// motion.)
__device__ __forceinline__ void project_lane(const float (&q)[9], const float atD, const float atH, const float gamma,
                                             const float4 (&b)[4], float (&d)[4][3], float2& lam)
{
    float D[3][3];
#pragma unroll
    for (int i = 0; i < 3; i++) {
        D[i][0] = (b[i].x - b[3].x) + (d[i][0] - d[3][0]);
        D[i][1] = (b[i].y - b[3].y) + (d[i][1] - d[3][1]);
        D[i][2] = (b[i].z - b[3].z) + (d[i][2] - d[3][2]);
    }
    float F[9];
#pragma unroll
    for (int c = 0; c < 3; c++)
#pragma unroll
        for (int r = 0; r < 3; r++) {
            const float sum = sum_of_products(D[0][r], q[3 * c], D[1][r], q[3 * c + 1], D[2][r], q[3 * c + 2]);
            F[3 * c + r] = r == c ? sum + 1.f : sum;
        }
    float ss = fmaf(F[0], F[0], F[1] * F[1]);
#pragma unroll
    for (int i = 2; i < 9; i++) ss = fmaf(F[i], F[i], ss);
    const float CD = xsqrt<float>(ss);
    auto cross = [](float p, float r, float s, float t) { return fmaf(p, r, -(s * t)); };
    float Fc[9];
    Fc[0] = cross(F[4], F[8], F[5], F[7]);
    Fc[1] = cross(F[5], F[6], F[3], F[8]);
    Fc[2] = cross(F[3], F[7], F[4], F[6]);
    Fc[3] = cross(F[7], F[2], F[8], F[1]);
    Fc[4] = cross(F[8], F[0], F[6], F[2]);
    Fc[5] = cross(F[6], F[1], F[7], F[0]);
    Fc[6] = cross(F[1], F[5], F[2], F[4]);
    Fc[7] = cross(F[2], F[3], F[0], F[5]);
    Fc[8] = cross(F[0], F[4], F[1], F[3]);
    const float J = sum3(F[0], Fc[0], F[1], Fc[1], F[2], Fc[2]);
    const float a = J - 1.f, aa = a * a;
    const float ch_log = -gamma + xlog<float>(J);
    const float ch_series = fmaf(aa * a, 1.f / 3.f, fmaf(aa, -0.5f, a - gamma));
    const float CH = J >= 1.f ? ch_log : ch_series;
    const float inv_C = xrcp<float>(CD);
    const float fac = (J >= 1.f) ? xrcp<float>(J) : fmaf(a, a, 1.f - a);
    float gD[4][3], gH[4][3], w[4], dd[4], dh[4], hh[4];
#pragma unroll
    for (int j = 0; j < 4; j++) {
        float qj[3];
#pragma unroll
        for (int c = 0; c < 3; c++) qj[c] = j < 3 ? q[3 * c + j] : -(q[3 * c] + q[3 * c + 1] + q[3 * c + 2]);
#pragma unroll
        for (int r = 0; r < 3; r++) {
            gD[j][r] = inv_C * sum3(F[r], qj[0], F[3 + r], qj[1], F[6 + r], qj[2]);
            gH[j][r] = fac * sum3(Fc[r], qj[0], Fc[3 + r], qj[1], Fc[6 + r], qj[2]);
        }
        w[j] = b[j].w;
        dd[j] = sum3(gD[j][0], gD[j][0], gD[j][1], gD[j][1], gD[j][2], gD[j][2]);
        dh[j] = sum3(gD[j][0], gH[j][0], gD[j][1], gH[j][1], gD[j][2], gH[j][2]);
        hh[j] = sum3(gH[j][0], gH[j][0], gH[j][1], gH[j][1], gH[j][2], gH[j][2]);
    }
    const float A01 = sum_of_products(w, dh);
    const float A00 = atD + sum_of_products(w, dd), A11 = atH + sum_of_products(w, hh);
    const float b0 = fmaf(-atD, lam.x, -CD), b1 = fmaf(-atH, lam.y, -CH);
    // a non-positive FP32 determinant (slivers) skips the projection, as in project_tet_F
    const float det = cross(A00, A11, A01, A01);
    const float inv_det = det > 0.f ? xrcp<float>(det) : 0.f;
    const float n0 = cross(b0, A11, b1, A01), n1 = cross(b1, A00, b0, A01);
    const float d0 = n0 * inv_det, d1 = n1 * inv_det;
    lam.x = fmaf(n0, inv_det, lam.x);
    lam.y = fmaf(n1, inv_det, lam.y);
#pragma unroll
    for (int j = 0; j < 4; j++)
#pragma unroll
        for (int k = 0; k < 3; k++) d[j][k] = fmaf(w[j], fmaf(gD[j][k], d0, gH[j][k] * d1), d[j][k]);
}

// The tile kernel with one lane a cluster: 64 clusters a block, N rows each
// (a cluster with fewer elements has empty ones: no weights, the slot that
// stands for no vertex).  RING rows are in flight ahead of the one projected.
// CAP: more slots than a tile has; the motions lie CAP * 16 bytes behind the
// bases, a distance that LDS instructions hold themselves.
template <int N, int RING, int CAP, bool IMPORT>
__global__ __launch_bounds__(512) void k_gs_tile_lane(GsTileArgs A)
{
    static_assert(N % RING == 0, "a row's place in the ring does not change from block to block");
    static_assert(CAP < 4096, "slot offsets are 16 bits, and so are LDS instructions' own");
    extern __shared__ float4 lds[];
    char* const lb = reinterpret_cast<char*>(lds);   // base, inverse mass; then in-step motion
    const int lane = threadIdx.x & 63;
    const int t = xcd_item(blockIdx.x, gridDim.x, true);
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const size_t tw = (size_t)t * A.waves + min(wave, A.waves - 1);   // waves past the last only stage
    const int2 tile = A.tile[t], head = A.wave[tw];
    const int* list = A.list + tw * A.blocks;
    int cur = list[0], nxt = list[min(1, A.blocks - 1)];
    TileStage<kStageLane> g;
    tile_load(A, t, threadIdx.x, g);
    __builtin_amdgcn_sched_barrier(0);   // these return first
    // a row: Q (9), alpha tilde D, H, gamma; four 16-bit slots (as byte offsets)
    float4 S[RING][3];
    uint2 V[RING];
    float2 L[RING];
    const float4* const st0 = A.stream + tw * A.rows * kLaneRow + lane;
    const uint2* const sv0 = reinterpret_cast<const uint2*>(A.stream + tw * A.rows * kLaneRow + 192) + lane;
    float2* const sl0 = A.lam + tw * A.rows * 64 + lane;
    const int* home = A.home + tw * A.blocks * 64 + lane;   // 2 * first solver position + whether this copy writes dlam
    const float4* st = st0;   // the next row to load
    const uint2* sv = sv0;
    auto load_row = [&](const float2* sl, int k, int c) {
#pragma unroll
        for (int p = 0; p < 3; p++) S[c][p] = st[p * 64];
        V[c] = *sv;
        if (!IMPORT) L[c] = sl[k * 64];
        st += kLaneRow;
        sv += 2 * kLaneRow;
    };
    int H = 0;
    const int nb = wave < A.waves ? head.x : 0;
    auto first_rows = [&] {
        H = home[0];
#pragma unroll
        for (int k = 0; k < RING; k++) load_row(sl0, k, k);
    };
    // the rows of the first phase arrive with the slots, those of later phases
    // after them: all workgroups start at once, and what they ask for together
    // is as much as the memory gives in several microseconds
    if (nb > 0 && head.y == 0) first_rows();
    __builtin_amdgcn_sched_barrier(0);
    tile_stage(A, t, g, [&](int i, const float4 b, const float4 d) {
        *reinterpret_cast<float4*>(lb + 16 * i) = b;
        *reinterpret_cast<float4*>(lb + 16 * CAP + 16 * i) = d;
    });
    lds_barrier();
    if (nb > 0 && head.y > 0) first_rows();
    const TileOut to = tile_out(A, t);
    if (nb == 0) {
        for (int i = A.niter * tile.x; i > 0; i--) lds_barrier();
    } else {
        // slots and bases of the row to come: they do not wait for the one before it
        uint32_t v[4];
        float4 b[4];
        auto load_base = [&](int c) {
            const uint32_t i01 = V[c].x, i23 = V[c].y;
            v[0] = i01 & 0xffffu;
            v[1] = i01 >> 16;
            v[2] = i23 & 0xffffu;
            v[3] = i23 >> 16;
#pragma unroll
            for (int m = 0; m < 4; m++) b[m] = *reinterpret_cast<const float4*>(lb + v[m]);
        };
        load_base(0);
        if (nb == 1) nxt = cur;
        for (int it = 0; it < A.niter; it++) {
            const bool out = A.lam_out && it == A.niter - 1;
            const bool zero = !IMPORT && it == 0 && A.lam_zero;
            for (int i = head.y; i > 0; i--) lds_barrier();
            float2* sl = sl0;
            for (int i = 0; i < nb; i++) {
                const int ent = __builtin_amdgcn_readfirstlane(nxt);
                nxt = list[i + 2 < nb ? i + 2 : min(i + 2 - nb, nb - 1)];
                const bool wrap = i + 1 == nb;
                const int Hn = home[wrap ? 0 : (i + 1) * 64];
                float2* const sln = wrap ? sl0 : sl + N * 64;
#pragma unroll
                for (int k = 0; k < N; k++) {
                    const int c = k % RING;
                    const float4 e0 = S[c][0], e1 = S[c][1], e2 = S[c][2];
                    const float q[9] = { e0.x, e0.y, e0.z, e0.w, e1.x, e1.y, e1.z, e1.w, e2.x };
                    float2 l = L[c];
                    if (zero) l = make_float2(0.f, 0.f);
                    if (IMPORT) l = A.kept[min((H >> 1) + k, A.nt - 1)];
                    uint32_t u[4];
                    float4 bb[4], f[4];
#pragma unroll
                    for (int m = 0; m < 4; m++) {
                        u[m] = v[m];
                        bb[m] = b[m];
                        f[m] = *reinterpret_cast<const float4*>(lb + u[m] + 16 * CAP);
                    }
                    load_base((k + 1) % RING);
                    float d[4][3];
#pragma unroll
                    for (int m = 0; m < 4; m++) {
                        d[m][0] = f[m].x;
                        d[m][1] = f[m].y;
                        d[m][2] = f[m].z;
                    }
                    project_lane(q, e2.y, e2.z, e2.w, bb, d, l);
#pragma unroll
                    for (int m = 0; m < 4; m++)
                        *reinterpret_cast<float4*>(lb + u[m] + 16 * CAP) = make_float4(d[m][0], d[m][1], d[m][2], 0.f);
                    sl[k * 64] = l;
                    if (out) {
                        if ((H & 1) && u[0] != 16u * (A.slots - 1)) A.dlam[(H >> 1) + k] = l;
                    }
                    if (k + RING == N && wrap) {
                        st = st0;
                        sv = sv0;
                    }
                    load_row(k + RING < N ? sl : sln, k + RING < N ? k + RING : k + RING - N, c);
                }
                for (int n = cur >> 4; n > 0; n--) lds_barrier();
                cur = ent;
                H = Hn;
                sl = sln;
            }
        }
    }
    tile_write(A, to, t, tile.y, [&](int i) { return *reinterpret_cast<const float4*>(lb + 16 * CAP + 16 * i); });
}

// Lays out a group's element data for k_gs_tile_lane: a thread per cluster copy.
__global__ __launch_bounds__(256) void k_gs_tile_lane_fill(GsTileFill A)
{
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i >= A.nblocks * 64) return;
    const int b = i >> 6, lane = i & 63;
    const int c = A.clu[i];
    const int e0 = c >= 0 ? A.cstart[c] : 0, n = c >= 0 ? A.cstart[c + 1] - e0 : 0;
    A.home[i] = 2 * e0 + (A.own[i] ? 1 : 0);
    const int rows = A.list[b] & 15;
    const size_t row = (size_t)A.row[b];
    for (int k = 0; k < rows; k++) {
        float f[12];
        for (int m = 0; m < 12; m++) f[m] = 0.f;
        uint32_t v[4];
        for (int m = 0; m < 4; m++) v[m] = (uint32_t)(A.slots - 1);
        if (k < n) {
            const int e = e0 + k;
            for (int m = 0; m < 9; m++) f[m] = A.ta.Q[(size_t)m * A.ta.qstride + e];
            const float2 at = A.ta.at[e];
            f[9] = at.x;
            f[10] = at.y;
            f[11] = A.ta.gamma[e];
            for (int m = 0; m < 4; m++) v[m] = A.vert[(size_t)i * 8 + ((A.tloc[e] >> (4 * m)) & 15u)];
        }
        float4* const st = A.stream + (row + k) * kLaneRow;
        for (int p = 0; p < 3; p++) st[p * 64 + lane] = make_float4(f[4 * p], f[4 * p + 1], f[4 * p + 2], f[4 * p + 3]);
        reinterpret_cast<uint2*>(st + 192)[lane] = make_uint2(16 * v[0] | v[1] << 20, 16 * v[2] | v[3] << 20);
        A.lam[(row + k) * 64 + lane] = make_float2(0.f, 0.f);
    }
}

// The step's motions and bases out of the vertex records into all groups' slots
// (the motions into the first group's, whose slots come first), and the motions
// back from the owners' slots.  PREDICT: the motions are the step's prediction,
// formed here, and the launch makes the lists of a detection's hits too.
template <bool PREDICT>
__global__ __launch_bounds__(256) void k_gs_tile_load(const float4* __restrict__ pos, const int* __restrict__ slot_vert,
                                                     int n, int nd, float4* __restrict__ d, float4* __restrict__ base,
                                                     Prediction P, HitLists H, int nload)
{
    if constexpr (PREDICT) {
        __shared__ int ws[2 * kStepWaves];
        if ((int)blockIdx.x >= nload) {
            scatter_hits(H, blockIdx.x - nload, gridDim.x - nload, ws);
            return;
        }
    }
    const int s = blockIdx.x * 256 + threadIdx.x;
    if (s >= n) return;
    const int v = slot_vert[s];
    float4 b = make_float4(0.f, 0.f, 0.f, 0.f), x = b;
    if (v >= 0) {
        b = pos[2 * (size_t)v];
        if (s < nd) x = PREDICT ? predicted(P, v) : pos[2 * (size_t)v + 1];
    }
    base[s] = b;
    if (s < nd) d[s] = x;
}
__global__ __launch_bounds__(256) void k_gs_tile_store(float4* __restrict__ pos, const int* __restrict__ owner, int nv,
                                                      const float4* __restrict__ d)
{
    const int v = blockIdx.x * 256 + threadIdx.x;
    if (v < nv) pos[2 * (size_t)v + 1] = d[owner[v]];
}

}  // namespace

size_t gs_tile_smem(int slots, const GsTileShape& S)
{
    return S.lanes == 1 ? 16 * ((size_t)S.cap + slots) : 28 * (size_t)slots;
}

int gs_tile_cap(int slots)
{
    for (int c : { 1024, 2048, 4095 })
        if (slots <= c) return c;
    return 0;
}

namespace {
typedef void (*TileKernel)(GsTileArgs);
template <int N, int RING, bool IMPORT>
TileKernel lane_kernel(int cap)
{
    return cap <= 1024   ? k_gs_tile_lane<N, RING, 1024, IMPORT>
           : cap <= 2048 ? k_gs_tile_lane<N, RING, 2048, IMPORT>
                         : k_gs_tile_lane<N, RING, 4095, IMPORT>;
}
TileKernel tile_kernel(const GsTileShape& S, bool import)
{
    if (S.lanes == 1) {
        if (S.rows == 8) return import ? lane_kernel<8, 4, true>(S.cap) : lane_kernel<8, 4, false>(S.cap);
        return import ? lane_kernel<6, 3, true>(S.cap) : lane_kernel<6, 3, false>(S.cap);
    }
    if (S.rows > 6) return import ? k_gs_tile<8, false, true> : k_gs_tile<8, false, false>;
    if (S.full) return import ? k_gs_tile<6, true, true> : k_gs_tile<6, true, false>;
    return import ? k_gs_tile<6, false, true> : k_gs_tile<6, false, false>;
}
}  // namespace

// The limit is the kernel's, not a handle's: always the most a plan may ask for.
hipError_t gs_tile_prepare(const GsTileShape& S)
{
    hipError_t e = hipSuccess;
    for (int i = 0; i < 2 && e == hipSuccess; i++)
        e = hipFuncSetAttribute(reinterpret_cast<const void*>(tile_kernel(S, i != 0)),
                                hipFuncAttributeMaxDynamicSharedMemorySize, (int)kGsTileLds);
    return e;
}

hipError_t launch_gs_tile(hipStream_t s, const GsTileArgs& A, const GsTileShape& S, int ntiles, int threads, size_t smem,
                          bool import)
{
    if (ntiles <= 0 || A.niter <= 0) return hipSuccess;
    if (threads < 64 || threads > (S.lanes == 1 ? 512 : 1024) || threads % 64) return hipErrorInvalidValue;
    hipLaunchKernelGGL(tile_kernel(S, import), dim3(ntiles), dim3(threads), smem, s, A);
    return hipGetLastError();
}

hipError_t launch_gs_tile_fill(hipStream_t s, const GsTileFill& A, const GsTileShape& S)
{
    if (A.nblocks <= 0) return hipSuccess;
    const dim3 g((unsigned)((A.nblocks + 3) / 4));
    if (S.lanes == 1) hipLaunchKernelGGL(k_gs_tile_lane_fill, g, dim3(256), 0, s, A);
    else hipLaunchKernelGGL(k_gs_tile_fill, g, dim3(256), 0, s, A);
    return hipGetLastError();
}

hipError_t launch_gs_tile_load(hipStream_t s, const float4* pos, const int* slot_vert, int n, int nd, float4* d,
                               float4* base, const Prediction* predict, const HitLists* hits)
{
    const int nl = (n + 255) / 256, nh = hits && hits->nf > 0 ? compact_blocks(hits->nf) : 0;
    if (nl + nh <= 0) return hipSuccess;
    if (hits && !predict) return hipErrorInvalidValue;
    if (predict)
        hipLaunchKernelGGL(k_gs_tile_load<true>, dim3(nl + nh), dim3(256), 0, s, pos, slot_vert, n, nd, d, base, *predict,
                           hits ? *hits : HitLists{}, nl);
    else
        hipLaunchKernelGGL(k_gs_tile_load<false>, dim3(nl), dim3(256), 0, s, pos, slot_vert, n, nd, d, base, Prediction{},
                           HitLists{}, nl);
    return hipGetLastError();
}

hipError_t launch_gs_tile_store(hipStream_t s, float4* pos, const int* owner, int nv, const float4* d)
{
    if (nv <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_gs_tile_store, dim3((unsigned)((nv + 255) / 256)), dim3(256), 0, s, pos, owner, nv, d);
    return hipGetLastError();
}

}  // namespace xpbd
