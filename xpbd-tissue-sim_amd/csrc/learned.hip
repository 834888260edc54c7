// Learned warm start: a 24 -> 128 -> 128 -> 3 per-vertex MLP (SiLU) whose
// GEMMs run on gfx950 BF16 MFMA (v_mfma_f32_16x16x32_bf16) with FP32
// accumulation, trained on the device with Adam, and the learned solver step.
//
// MFMA 16x16x32 operand layout (wave64, lane l):
//   A (16 x 32, M x K): row l % 16, k = 8 * (l / 16) + 0..7
//   B (32 x 16, K x N): col l % 16, k = 8 * (l / 16) + 0..7
//   D (16 x 16):        col l % 16, rows 4 * (l / 16) + 0..3
//
// The learned step (no counterpart in the reference): after the inertial
// prediction x~, the network predicts the solver's correction c; the solve
// starts at x0 = x~ + c with the multipliers that satisfy the constraint
// equations there, lambda0 = -C(x0) / alpha~, and runs the configured number
// of Gauss-Seidel / Jacobi iterations (which resolve contacts and whatever the
// network did not predict).  If the constraint residual then exceeds
// ratio * reference, the step is redone from the saved state with the plain
// cold-start solve (the reference solver's semantics).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <cmath>
#include <cstdio>
#include <cstring>
#include <mutex>
#include <new>
#include <random>
#include <string>
#include <vector>

#include "capi_internal.h"
#include "kernels.h"
#include "step_ops.h"
#include "xpbd_math.h"

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

namespace {

constexpr int kIn = XPBD_MLP_IN, kInP = 32, kH = XPBD_MLP_HIDDEN, kOut = XPBD_MLP_OUT, kOutP = 16;
// parameter offsets in the FP32 master vector
constexpr int oW1 = 0, oB1 = oW1 + kH * kIn, oW2 = oB1 + kH, oB2 = oW2 + kH * kH, oW3 = oB2 + kH,
              oB3 = oW3 + kOut * kH, kNParams = oB3 + kOut;
static_assert(kNParams == 20099, "parameter count");

__device__ __forceinline__ float silu(float z) { return z / (1.0f + __expf(-z)); }
// inference: hardware reciprocal (1 ulp) in place of the IEEE division; the
// result is rounded to BF16 right after
__device__ __forceinline__ float silu_fast(float z) { return z * __builtin_amdgcn_rcpf(1.0f + __expf(-z)); }
__device__ __forceinline__ float dsilu(float z)
{
    const float s = 1.0f / (1.0f + __expf(-z));
    return s * (1.0f + z * (1.0f - s));
}

// ---------------------------------------------------------------------------
// Training, three launches a minibatch.
//   rows     forward and back: a workgroup of 8 waves takes 32 rows, wave w the
//            hidden features 16w..16w+15 of every layer, so that the pre-activations
//            stay in its registers and only the activations and their gradients go
//            through LDS, as the BF16 A operand of the next product.  Weights are B
//            operands, read once from a copy in operand order that the update keeps
//            beside the FP32 master.  Activations (BF16) and gradients (FP32) are
//            left feature by feature, a lane's four rows together.
//   weights  the weight gradients' products, whose K is the rows, by runs of rows,
//            and the bias gradients' column sums
//   update   sums of the runs in order, Adam, the weights' operand copies
// Every sum is formed in the order of a plain product by 32 rows at a time with its
// runs of rows added up in turn, whatever the grid: a last bit that differs can round
// an activation to another BF16 number, and over some epochs that shows.
//
// 4,096 rows: 24 launches before, 175 us with the update, now 13.5 + 9.8 + 3.7 us in three.  Bound by the
// chain of a tile of rows: five small products, a barrier after each, and the SiLUs'
// divisions between.
// ---------------------------------------------------------------------------
constexpr int kTrainRows = 32, kTrainWaves = kH / 16, kTrainThreads = 64 * kTrainWaves;
// operand copies of the weights: products of 64 lanes x 8 values
constexpr int kK2 = kH / 32;   // K steps over the hidden features
constexpr int fW1 = 0, fW2 = fW1 + kTrainWaves, fW2T = fW2 + kTrainWaves * kK2, fW3 = fW2T + kTrainWaves * kK2,
              fW3T = fW3 + kK2, kFrags = fW3T + kTrainWaves;

// The places of parameter i among the operand copies (B operand of a product's
// step: column l % 16, k = 8 (l / 16) + 0..7), the second -1 if there is one only;
// both -1 for a bias.
__device__ __forceinline__ int2 operand_places(int i)
{
    auto at = [](int f, int col, int k) { return 512 * f + 8 * (col + 16 * (k >> 3)) + (k & 7); };
    if (i < oB1) {
        const int o = i / kIn, k = i % kIn;
        return make_int2(at(fW1 + o / 16, o % 16, k), -1);
    }
    if (i >= oW2 && i < oB2) {
        const int o = (i - oW2) / kH, k = (i - oW2) % kH;
        return make_int2(at(fW2 + o / 16 * kK2 + k / 32, o % 16, k % 32), at(fW2T + k / 16 * kK2 + o / 32, k % 16, o % 32));
    }
    if (i >= oW3 && i < oB3) {
        const int o = (i - oW3) / kH, k = (i - oW3) % kH;
        return make_int2(at(fW3 + k / 32, o, k % 32), at(fW3T + k / 16, k % 16, o));
    }
    return make_int2(-1, -1);
}

__device__ __forceinline__ void put_operand(__bf16* w, int i, float p)
{
    const int2 q = operand_places(i);
    if (q.x >= 0) w[q.x] = (__bf16)p;
    if (q.y >= 0) w[q.y] = (__bf16)p;
}

// all operand copies from the master (what no parameter has a place in was zeroed when the copies were made)
__global__ void k_train_pack(const float* __restrict__ p, __bf16* __restrict__ w)
{
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i < kNParams) put_operand(w, i, p[i]);
}

__device__ __forceinline__ void put4(__bf16* dst, const float* v)
{
    typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
    *reinterpret_cast<bf16x4*>(dst) = bf16x4{ (__bf16)v[0], (__bf16)v[1], (__bf16)v[2], (__bf16)v[3] };
}

__device__ __forceinline__ f32x4 mfma(bf16x8 a, bf16x8 b, f32x4 c)
{
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}

// A minibatch's activations and gradients, feature by feature: ld values (its rows up
// to a multiple of 32, zero gradients past them) each.
struct TrainRows {
    int ld = 0;
    __bf16 *x = nullptr, *h1 = nullptr, *h2 = nullptr;           // kInP, kH, kH features
    float *d1 = nullptr, *d2 = nullptr, *dy = nullptr;           // kH, kH, kOut
    double* loss = nullptr;                                      // per 32 rows

    static size_t bytes(size_t ld) { return ld * (2 * (kInP + 2 * kH) + 4 * (2 * kH + kOut)) + 8 * (ld / kTrainRows); }
    void place(char* p, int rows)
    {
        ld = rows;
        const size_t n = (size_t)rows;
        d1 = reinterpret_cast<float*>(p);
        d2 = d1 + kH * n;
        dy = d2 + kH * n;
        x = reinterpret_cast<__bf16*>(dy + kOut * n);
        h1 = x + kInP * n;
        h2 = h1 + kH * n;
        loss = reinterpret_cast<double*>(h2 + kH * n);
    }
};

// Row r of the minibatch is row perm[(b0 + r) % nall] of X and T (perm null: r).
// Loss in output units of the network: mean over rows * 3 of (Y - T / scale)^2,
// i.e. the squared error of the correction measured in units of scale (the
// physical corrections are ~1e-5 m; a loss in metres would leave gradients far
// below Adam's epsilon).  dY = 2 (Y - T / scale) / (rows * 3).
__global__ __launch_bounds__(kTrainThreads) void k_train_rows(const float* __restrict__ X, const float* __restrict__ T,
                                                             const int* __restrict__ perm, int b0, int nall, int rows,
                                                             const float* __restrict__ mean,
                                                             const float* __restrict__ istd, float inv_scale,
                                                             const float* __restrict__ p, const __bf16* __restrict__ w,
                                                             TrainRows out)
{
    constexpr int R = kTrainRows, LR = R + 8, LH = kH + 8;   // padded: rows of 16-byte multiples, banks apart
    __shared__ alignas(16) __bf16 aX[R][LR], aH1[R][LH], aH2[R][LH], aD2[R][LH], aY[R][LR];
    __shared__ float sT[R][4];
    __shared__ double sl[2 * 64];
    const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6, c = lane & 15, q = lane >> 4;
    const int col = 16 * wv + c, r0 = blockIdx.x * R;   // col: this lane's hidden feature
    auto frag = [&](int f) { return reinterpret_cast<const bf16x8*>(w)[64 * f + lane]; };
    const bf16x8 w1 = frag(fW1 + wv), w3t = frag(fW3T + wv);
    bf16x8 w2[kK2], w2t[kK2], w3[kK2];
#pragma unroll
    for (int k = 0; k < kK2; k++) {
        w2[k] = frag(fW2 + wv * kK2 + k);
        w2t[k] = frag(fW2T + wv * kK2 + k);
        w3[k] = frag(fW3 + k);
    }
    const float b1 = p[oB1 + col], b2 = p[oB2 + col], b3 = c < kOut ? p[oB3 + c] : 0.f;
    const f32x4 zero = { 0.f, 0.f, 0.f, 0.f };
    for (int i = tid; i < R * LR; i += kTrainThreads) aY[i / LR][i % LR] = (__bf16)0.f;   // its columns 16.. stay zero
    for (int i = tid; i < R * kInP; i += kTrainThreads) {
        const int r = i / kInP, k = i % kInP;
        float x = 0.f;
        if (r0 + r < rows) {
            const int src = perm ? perm[(b0 + r0 + r) % nall] : r0 + r;
            if (k < kIn) x = (X[(size_t)src * kIn + k] - mean[k]) * istd[k];
            else if (k < kIn + kOut) sT[r][k - kIn] = T[(size_t)src * kOut + k - kIn];
        }
        aX[r][k] = (__bf16)x;
        out.x[(size_t)k * out.ld + r0 + r] = (__bf16)x;
    }
    __syncthreads();
    // this lane's rows of feature f among those left: 16 m + 4q + 0..3
    auto at = [&](int f, int m) { return (size_t)f * out.ld + r0 + 16 * m + 4 * q; };
    // forward
    f32x4 z1[2], z2[2];
#pragma unroll
    for (int m = 0; m < 2; m++) {
        z1[m] = mfma(*reinterpret_cast<const bf16x8*>(&aX[16 * m + c][8 * q]), w1, zero);
        float h[4];
#pragma unroll
        for (int j = 0; j < 4; j++) {
            z1[m][j] += b1;
            h[j] = silu(z1[m][j]);
            aH1[16 * m + 4 * q + j][col] = (__bf16)h[j];
        }
        put4(out.h1 + at(col, m), h);
    }
    __syncthreads();
#pragma unroll
    for (int m = 0; m < 2; m++) {
        z2[m] = zero;
#pragma unroll
        for (int k = 0; k < kK2; k++)
            z2[m] = mfma(*reinterpret_cast<const bf16x8*>(&aH1[16 * m + c][32 * k + 8 * q]), w2[k], z2[m]);
        float h[4];
#pragma unroll
        for (int j = 0; j < 4; j++) {
            z2[m][j] += b2;
            h[j] = silu(z2[m][j]);
            aH2[16 * m + 4 * q + j][col] = (__bf16)h[j];
        }
        put4(out.h2 + at(col, m), h);
    }
    __syncthreads();
    // output and its gradient: waves 0 and 1, 16 rows each
    if (wv < 2) {
        f32x4 y = zero;
#pragma unroll
        for (int k = 0; k < kK2; k++)
            y = mfma(*reinterpret_cast<const bf16x8*>(&aH2[16 * wv + c][32 * k + 8 * q]), w3[k], y);
        float d[4];
        double loss = 0.0;
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const int r = 16 * wv + 4 * q + j;
            const bool on = c < kOut && r0 + r < rows;
            const float e = on ? fmaf(-sT[r][c & 3], inv_scale, y[j] + b3) : 0.f;
            d[j] = on ? 2.0f * e / (float)(rows * kOut) : 0.f;
            loss += (double)e * (double)e;
            aY[r][c] = (__bf16)d[j];
        }
        if (c < kOut) *reinterpret_cast<float4*>(out.dy + at(c, wv)) = make_float4(d[0], d[1], d[2], d[3]);
        sl[64 * wv + lane] = loss;
    }
    __syncthreads();
    // back through layer 3
#pragma unroll
    for (int m = 0; m < 2; m++) {
        const f32x4 h = mfma(*reinterpret_cast<const bf16x8*>(&aY[16 * m + c][8 * q]), w3t, zero);
        float d[4];
#pragma unroll
        for (int j = 0; j < 4; j++) {
            d[j] = h[j] * dsilu(z2[m][j]);
            aD2[16 * m + 4 * q + j][col] = (__bf16)d[j];
        }
        *reinterpret_cast<float4*>(out.d2 + at(col, m)) = make_float4(d[0], d[1], d[2], d[3]);
    }
    if (tid == 0) {
        double l = 0.0;
        for (int i = 0; i < 2 * 64; i++) l += sl[i];
        out.loss[blockIdx.x] = l;
    }
    __syncthreads();
    // and layer 2
#pragma unroll
    for (int m = 0; m < 2; m++) {
        f32x4 h = zero;
#pragma unroll
        for (int k = 0; k < kK2; k++)
            h = mfma(*reinterpret_cast<const bf16x8*>(&aD2[16 * m + c][32 * k + 8 * q]), w2t[k], h);
        float d[4];
#pragma unroll
        for (int j = 0; j < 4; j++) d[j] = h[j] * dsilu(z1[m][j]);
        *reinterpret_cast<float4*>(out.d1 + at(col, m)) = make_float4(d[0], d[1], d[2], d[3]);
    }
}

// Runs of rows that a weight gradient of `tiles` output tiles of 32 x 32 is formed
// by: of at least 128 rows, up to 512 tiles' worth and kMaxRuns of them.
constexpr int kMaxRuns = 64, kRuns2 = 32;
struct Runs {
    int rows, n;
};
inline Runs runs_of(int rows, int tiles)
{
    int n = 1;
    if (rows >= 256) n = std::min(std::min((512 + tiles - 1) / tiles, (rows + 127) / 128), kMaxRuns);
    const int len = ((rows + n - 1) / n + 31) / 32 * 32;
    return { len, (rows + len - 1) / len };
}

// eight rows of one feature's gradient as an operand
__device__ __forceinline__ bf16x8 as_operand(const float* d)
{
    const float4 a = reinterpret_cast<const float4*>(d)[0], b = reinterpret_cast<const float4*>(d)[1];
    return bf16x8{ (__bf16)a.x, (__bf16)a.y, (__bf16)a.z, (__bf16)a.w, (__bf16)b.x, (__bf16)b.y, (__bf16)b.z, (__bf16)b.w };
}

// Blocks 4 z + k: rows 32k..32k+31 of layer 2's weight gradient over run z of r2; then
// one a run of r13 for layers 1 and 3; then one a bias.  A wave has 16 x 64 outputs of
// layer 2 (32 x 32 of layer 1, 16 x 32 of layer 3), 32 rows of the minibatch a step.
__global__ __launch_bounds__(256) void k_train_weights(TrainRows in, int rows, Runs r2, Runs r13,
                                                      float* __restrict__ part2, float* __restrict__ part13,
                                                      float* __restrict__ bias)
{
    const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6, c = lane & 15, q = lane >> 4;
    const size_t ld = (size_t)in.ld;
    const f32x4 zero = { 0.f, 0.f, 0.f, 0.f };
    int b = blockIdx.x;
    if (b < 4 * r2.n) {
        const int z = b >> 2, o0 = 32 * (b & 3) + 16 * (wv >> 1), i0 = 64 * (wv & 1);
        const int k0 = z * r2.rows, k1 = min(rows, k0 + r2.rows);
        f32x4 g[4] = { zero, zero, zero, zero };
#pragma unroll 4
        for (int k = k0; k < k1; k += 32) {
            const bf16x8 d = as_operand(in.d2 + (o0 + c) * ld + k + 8 * q);
#pragma unroll
            for (int t = 0; t < 4; t++)
                g[t] = mfma(d, *reinterpret_cast<const bf16x8*>(in.h1 + (i0 + 16 * t + c) * ld + k + 8 * q), g[t]);
        }
        float* const o = part2 + (size_t)z * kH * kH;
#pragma unroll
        for (int t = 0; t < 4; t++)
#pragma unroll
            for (int j = 0; j < 4; j++) o[(o0 + 4 * q + j) * kH + i0 + 16 * t + c] = g[t][j];
        return;
    }
    b -= 4 * r2.n;
    if (b < r13.n) {
        const int k0 = b * r13.rows, k1 = min(rows, k0 + r13.rows);
        f32x4 g1[2][2] = { { zero, zero }, { zero, zero } }, g3[2] = { zero, zero };
#pragma unroll 2
        for (int k = k0; k < k1; k += 32) {
            bf16x8 y{};
            if (c < kOut) y = as_operand(in.dy + c * ld + k + 8 * q);
            bf16x8 x[2];
#pragma unroll
            for (int t = 0; t < 2; t++) x[t] = *reinterpret_cast<const bf16x8*>(in.x + (16 * t + c) * ld + k + 8 * q);
#pragma unroll
            for (int t = 0; t < 2; t++) {
                const int f = 32 * wv + 16 * t + c;
                const bf16x8 d = as_operand(in.d1 + f * ld + k + 8 * q);
                g1[t][0] = mfma(d, x[0], g1[t][0]);
                g1[t][1] = mfma(d, x[1], g1[t][1]);
                g3[t] = mfma(y, *reinterpret_cast<const bf16x8*>(in.h2 + f * ld + k + 8 * q), g3[t]);
            }
        }
        float* const o = part13 + (size_t)b * (kH * kIn + kOut * kH);
#pragma unroll
        for (int t = 0; t < 2; t++)
#pragma unroll
            for (int j = 0; j < 4; j++) {
                const int f = 32 * wv + 16 * t, row = 4 * q + j;
#pragma unroll
                for (int u = 0; u < 2; u++)
                    if (16 * u + c < kIn) o[(f + row) * kIn + 16 * u + c] = g1[t][u][j];
                if (row < kOut) o[kH * kIn + row * kH + f + c] = g3[t][j];
            }
        return;
    }
    b -= r13.n;   // a column sum: rows 256 apart by thread, then by halves
    __shared__ float sh[256];
    const float* d = b < kH ? in.d1 + b * ld : b < 2 * kH ? in.d2 + (b - kH) * ld : in.dy + (b - 2 * kH) * ld;
    float s = 0.f;
    for (int r = tid; r < rows; r += 256) s += d[r];
    sh[tid] = s;
    __syncthreads();
    for (int k = 128; k > 0; k >>= 1) {
        if (tid < k) sh[tid] += sh[tid + k];
        __syncthreads();
    }
    if (tid == 0) bias[b] = sh[0];
}

// The sum of the runs, in order, and with ADAM the update of the master, the moments
// and the operand copies; otherwise into g.
template <bool ADAM>
__global__ __launch_bounds__(256) void k_train_update(const float* __restrict__ part2, int n2,
                                                     const float* __restrict__ part13, int n13,
                                                     const float* __restrict__ bias, float* __restrict__ g,
                                                     float* __restrict__ p, float* __restrict__ m,
                                                     float* __restrict__ v, __bf16* __restrict__ w, float lr, float b1,
                                                     float b2, float c1, float c2, float eps)
{
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i >= kNParams) return;
    float gi = 0.f;
    const float* part = nullptr;
    size_t stride = kH * kIn + kOut * kH;
    int n = n13;
    if (i < oB1) part = part13 + i;
    else if (i < oW2) gi = bias[i - oB1];
    else if (i < oB2) {
        part = part2 + (i - oW2);
        stride = kH * kH;
        n = n2;
    } else if (i < oW3) gi = bias[kH + i - oB2];
    else if (i < oB3) part = part13 + kH * kIn + (i - oW3);
    else gi = bias[2 * kH + i - oB3];
    if (part) {
#pragma unroll 16
        for (int z = 0; z < n; z++) gi += part[z * stride];
    }
    if constexpr (!ADAM) {
        g[i] = gi;
        return;
    }
    const float mi = b1 * m[i] + (1.f - b1) * gi;
    const float vi = b2 * v[i] + (1.f - b2) * gi * gi;
    m[i] = mi;
    v[i] = vi;
    const float pi = p[i] - lr * (mi / c1) / (sqrtf(vi / c2) + eps);
    p[i] = pi;
    put_operand(w, i, pi);
}

// The hidden feature at MFMA K position pos (0..31) of K block m in the
// inference kernel: the order in which a 16 x 16 output tile pair leaves the
// features in a lane (position 8q + i holds 4q + i of the block's first tile for
// i < 4, 4q + i - 4 of its second tile for i >= 4).
__host__ __device__ constexpr int mlp_k_feature(int m, int pos)
{
    return 32 * m + ((pos & 7) < 4 ? 4 * (pos >> 3) + (pos & 7) : 16 + 4 * (pos >> 3) + (pos & 7) - 4);
}

constexpr bool mlp_k_order_is_a_permutation()
{
    for (int m = 0; m < kH / 32; m++)
        for (int f = 32 * m; f < 32 * m + 32; f++) {
            int hits = 0;
            for (int pos = 0; pos < 32; pos++) hits += mlp_k_feature(m, pos) == f;
            if (hits != 1) return false;
        }
    return true;
}
static_assert(mlp_k_order_is_a_permutation(), "every hidden feature at exactly one K position");
// the inference kernel's shapes: one 32-wide K step for the inputs (8 per lane,
// lanes q < 3 full), 16-wide output tiles in pairs, at most 4 outputs (lanes q = 0)
static_assert(kInP == 32 && kIn % 8 == 0 && kIn <= kInP && kH % 32 == 0 && kOut <= 4 && kOutP == 16,
              "shapes of k_mlp_fused");

// FP32 master -> BF16 MFMA layouts of the inference kernel: W1 [128][32] (k >= 24
// zero), W2 [128][128] and W3 [16][128] (rows >= 3 zero) with their hidden K index
// in mlp_k_feature order
__global__ void k_pack(const float* __restrict__ p, __bf16* __restrict__ w1, __bf16* __restrict__ w2,
                       __bf16* __restrict__ w3)
{
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i < kH * kInP) {
        const int o = i / kInP, k = i % kInP;
        w1[i] = (__bf16)(k < kIn ? p[oW1 + o * kIn + k] : 0.f);
    }
    if (i < kH * kH) {
        const int o = i / kH, k = i % kH;
        w2[i] = (__bf16)p[oW2 + o * kH + mlp_k_feature(k / 32, k % 32)];
    }
    if (i < kOutP * kH) {
        const int o = i / kH, k = i % kH;
        w3[i] = (__bf16)(o < kOut ? p[oW3 + o * kH + mlp_k_feature(k / 32, k % 32)] : 0.f);
    }
}

// ---------------------------------------------------------------------------
// Fused inference, 4 waves per workgroup, 16 rows per wave per tile.  Every
// layer forms Z^T = W H^T: the weights (BF16, staged once per workgroup in LDS)
// are the MFMA's A operand and the activations its B operand.  A 16 x 16 output
// tile leaves lane (q = lane / 16, c = lane % 16) holding features 4q..4q+3 of
// row c, so the two tiles of a 32-wide K block hold, per lane, features
// 4q + {0..3} and 16 + 4q + {0..3} of the block: after bias and SiLU, rounded to
// BF16, they are the next layer's B operand as they lie, with that layer's
// weights packed in the same K order (mlp_k_feature).  The activations stay in
// registers from input to output; the first layer's B operand is read from the
// input rows directly (lane (q, c): features 8q..8q+7 of row c, zero past 24).
// out[r] (float4) = scale * MLP((x_r - mean) * istd) (* mask[r]), w = 0.
// ---------------------------------------------------------------------------
constexpr int kFwdRows = 64;

__global__ __launch_bounds__(256) void k_mlp_fused(const float* __restrict__ X, int n, const __bf16* __restrict__ w1,
                                                  const __bf16* __restrict__ w2, const __bf16* __restrict__ w3,
                                                  const float* __restrict__ params, const float* __restrict__ mean,
                                                  const float* __restrict__ istd, float scale,
                                                  float4* __restrict__ out, const float* __restrict__ mask)
{
    __shared__ alignas(16) __bf16 sw1[kH][kInP + 8];
    __shared__ alignas(16) __bf16 sw2[kH][kH + 8];
    __shared__ alignas(16) __bf16 sw3[kOutP][kH + 8];
    __shared__ alignas(16) float sb[2 * kH + kOutP];
    const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
    // weights in 16-byte pieces (8 BF16 values; rows are multiples of 8 long and
    // the padded LDS rows start on 16-byte boundaries)
    for (int i = tid; i < kH * kInP / 8; i += 256)
        *reinterpret_cast<bf16x8*>(&sw1[i / (kInP / 8)][8 * (i % (kInP / 8))]) = reinterpret_cast<const bf16x8*>(w1)[i];
    for (int i = tid; i < kH * kH / 8; i += 256)
        *reinterpret_cast<bf16x8*>(&sw2[i / (kH / 8)][8 * (i % (kH / 8))]) = reinterpret_cast<const bf16x8*>(w2)[i];
    for (int i = tid; i < kOutP * kH / 8; i += 256)
        *reinterpret_cast<bf16x8*>(&sw3[i / (kH / 8)][8 * (i % (kH / 8))]) = reinterpret_cast<const bf16x8*>(w3)[i];
    for (int i = tid; i < kH; i += 256) {
        sb[i] = params[oB1 + i];
        sb[kH + i] = params[oB2 + i];
    }
    if (tid < kOutP) sb[2 * kH + tid] = tid < kOut ? params[oB3 + tid] : 0.f;
    __syncthreads();
    // from here on the waves share only the weights and biases, which they read
    const int c = lane & 15, q = lane >> 4, kq = 8 * q;
    const bool xin = kq < kIn;   // lanes q < 3 hold input features, q = 3 the zero padding
    float xm[8], xs[8];
#pragma unroll
    for (int i = 0; i < 8; i++) {
        xm[i] = xin ? mean[kq + i] : 0.f;
        xs[i] = xin ? istd[kq + i] : 0.f;
    }
    const int ntile = (n + kFwdRows - 1) / kFwdRows;
    // the next tile's input features are loaded while the current tile is computed
    float4 xa = make_float4(0.f, 0.f, 0.f, 0.f), xb = xa;
    auto load_row = [&](int t) {
        const int r = t * kFwdRows + wv * 16 + c;
        xa = xb = make_float4(0.f, 0.f, 0.f, 0.f);
        if (xin && r < n) {
            const float4* x4 = reinterpret_cast<const float4*>(X + (size_t)r * kIn + kq);
            xa = x4[0];
            xb = x4[1];
        }
    };
    if ((int)blockIdx.x < ntile) load_row(blockIdx.x);
    for (int t = blockIdx.x; t < ntile; t += gridDim.x) {
        const int r = t * kFwdRows + wv * 16 + c;
        const float xv[8] = { xa.x, xa.y, xa.z, xa.w, xb.x, xb.y, xb.z, xb.w };
        bf16x8 h0;
#pragma unroll
        for (int i = 0; i < 8; i++) h0[i] = (__bf16)((xv[i] - xm[i]) * xs[i]);
        if (t + (int)gridDim.x < ntile) load_row(t + gridDim.x);
        // layer 1: 8 output tiles, one K step; K block m of layer 2 from tiles 2m, 2m + 1
        bf16x8 h1[kH / 32];
#pragma unroll
        for (int m = 0; m < kH / 32; m++) {
            const bf16x8 a0 = *reinterpret_cast<const bf16x8*>(&sw1[32 * m + c][kq]);
            const bf16x8 a1 = *reinterpret_cast<const bf16x8*>(&sw1[32 * m + 16 + c][kq]);
            const f32x4 z0 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a0, h0, f32x4{ 0.f, 0.f, 0.f, 0.f }, 0, 0, 0);
            const f32x4 z1 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a1, h0, f32x4{ 0.f, 0.f, 0.f, 0.f }, 0, 0, 0);
            const float4 b0 = *reinterpret_cast<const float4*>(&sb[32 * m + 4 * q]);
            const float4 b1 = *reinterpret_cast<const float4*>(&sb[32 * m + 16 + 4 * q]);
            h1[m] = bf16x8{ (__bf16)silu_fast(z0[0] + b0.x), (__bf16)silu_fast(z0[1] + b0.y),
                            (__bf16)silu_fast(z0[2] + b0.z), (__bf16)silu_fast(z0[3] + b0.w),
                            (__bf16)silu_fast(z1[0] + b1.x), (__bf16)silu_fast(z1[1] + b1.y),
                            (__bf16)silu_fast(z1[2] + b1.z), (__bf16)silu_fast(z1[3] + b1.w) };
        }
        // layer 2: 8 output tiles x 4 K steps
        f32x4 z2[kH / 16];
#pragma unroll
        for (int nt = 0; nt < kH / 16; nt++) z2[nt] = f32x4{ 0.f, 0.f, 0.f, 0.f };
#pragma unroll
        for (int m = 0; m < kH / 32; m++)
#pragma unroll
            for (int nt = 0; nt < kH / 16; nt++) {
                const bf16x8 a = *reinterpret_cast<const bf16x8*>(&sw2[nt * 16 + c][32 * m + kq]);
                z2[nt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, h1[m], z2[nt], 0, 0, 0);
            }
        bf16x8 h2[kH / 32];
#pragma unroll
        for (int m = 0; m < kH / 32; m++) {
            const float4 b0 = *reinterpret_cast<const float4*>(&sb[kH + 32 * m + 4 * q]);
            const float4 b1 = *reinterpret_cast<const float4*>(&sb[kH + 32 * m + 16 + 4 * q]);
            const f32x4 z0 = z2[2 * m], z1 = z2[2 * m + 1];
            h2[m] = bf16x8{ (__bf16)silu_fast(z0[0] + b0.x), (__bf16)silu_fast(z0[1] + b0.y),
                            (__bf16)silu_fast(z0[2] + b0.z), (__bf16)silu_fast(z0[3] + b0.w),
                            (__bf16)silu_fast(z1[0] + b1.x), (__bf16)silu_fast(z1[1] + b1.y),
                            (__bf16)silu_fast(z1[2] + b1.z), (__bf16)silu_fast(z1[3] + b1.w) };
        }
        // layer 3: one padded output tile x 4 K steps; lanes q = 0 hold outputs 0..3 of row c
        f32x4 y = { 0.f, 0.f, 0.f, 0.f };
#pragma unroll
        for (int m = 0; m < kH / 32; m++) {
            const bf16x8 a = *reinterpret_cast<const bf16x8*>(&sw3[c][32 * m + kq]);
            y = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, h2[m], y, 0, 0, 0);
        }
        if (q == 0 && r < n) {
            const float mk = mask ? mask[r] : 1.f;
            out[r] = make_float4(scale * (y[0] + sb[2 * kH]) * mk, scale * (y[1] + sb[2 * kH + 1]) * mk,
                                 scale * (y[2] + sb[2 * kH + 2]) * mk, 0.f);
        }
    }
}

inline unsigned nb(long long n) { return (unsigned)((n + 255) / 256); }

// out3[3 i + k] = out4[i].k for the first three components
__global__ void k_pack3(const float4* __restrict__ out4, int n, float* __restrict__ out3)
{
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i >= n) return;
    const float4 v = out4[i];
    out3[3 * (size_t)i] = v.x;
    out3[3 * (size_t)i + 1] = v.y;
    out3[3 * (size_t)i + 2] = v.z;
}

// ---------------------------------------------------------------------------
// solver-side kernels of the learned step
// ---------------------------------------------------------------------------
// Per-vertex features after the inertial prediction (row of 24 floats):
//   0-2   inertial displacement of this step (x~ - x)      3-5   velocity
//   6-8   1-ring mean of (u_j - u_i), u = x - X            9-11  1-ring mean of inertial displacement minus own
//   12-14 displacement from rest u_i                       15-17 previous step's solver correction c_i
//   18-20 1-ring mean of (c_j - c_i)                       21    mean log10 E of incident elements
//   22    mean nu of incident elements                     23    fraction of 1-ring neighbours pinned
__global__ void k_features(const float4* __restrict__ pos, const float4* __restrict__ vel,
                           const float4* __restrict__ cprev, const int* __restrict__ nb_off,
                           const int* __restrict__ nbr, const float2* __restrict__ vmat,
                           const float* __restrict__ pinfrac, int nv, float* __restrict__ feat)
{
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i >= nv) return;
    const float4 ui = pos[2 * (size_t)i], pi = pos[2 * (size_t)i + 1], vi = vel[i], ci = cprev[i];
    float su[3] = { 0.f, 0.f, 0.f }, sp[3] = { 0.f, 0.f, 0.f }, sc[3] = { 0.f, 0.f, 0.f };
    const int b = nb_off[i], e = nb_off[i + 1];
    for (int k = b; k < e; k++) {
        const int j = nbr[k];
        const float4 uj = pos[2 * (size_t)j], pj = pos[2 * (size_t)j + 1], cj = cprev[j];
        su[0] += uj.x; su[1] += uj.y; su[2] += uj.z;
        sp[0] += pj.x; sp[1] += pj.y; sp[2] += pj.z;
        sc[0] += cj.x; sc[1] += cj.y; sc[2] += cj.z;
    }
    const float inv = e > b ? 1.0f / (float)(e - b) : 0.f;
    const float own = e > b ? 1.f : 0.f;
    float* f = feat + (size_t)i * kIn;
    f[0] = pi.x; f[1] = pi.y; f[2] = pi.z;
    f[3] = vi.x; f[4] = vi.y; f[5] = vi.z;
    f[6] = su[0] * inv - own * ui.x; f[7] = su[1] * inv - own * ui.y; f[8] = su[2] * inv - own * ui.z;
    f[9] = sp[0] * inv - own * pi.x; f[10] = sp[1] * inv - own * pi.y; f[11] = sp[2] * inv - own * pi.z;
    f[12] = ui.x; f[13] = ui.y; f[14] = ui.z;
    f[15] = ci.x; f[16] = ci.y; f[17] = ci.z;
    f[18] = sc[0] * inv - own * ci.x; f[19] = sc[1] * inv - own * ci.y; f[20] = sc[2] * inv - own * ci.z;
    const float2 mt = vmat[i];
    f[21] = mt.x; f[22] = mt.y; f[23] = pinfrac[i];
}

// in-step motion after the prediction -> pred
__global__ void k_copy_delta(const float4* __restrict__ pos, float4* __restrict__ pred, int nv)
{
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i < nv) pred[i] = pos[2 * (size_t)i + 1];
}

// The start of a learned step in one launch: the state's snapshot for a fallback,
// the prediction and its copy, and the lists of a detection's hits, which were seven
// small launches and copies.
__global__ __launch_bounds__(xpbd::kStepBlock) void k_learned_begin(float4* __restrict__ pos,
                                                                   const float4* __restrict__ lo,
                                                                   const float4* __restrict__ vel, int nv,
                                                                   const unsigned long long* __restrict__ step,
                                                                   float4* __restrict__ save,
                                                                   unsigned long long* __restrict__ step_save,
                                                                   float4* __restrict__ pred, xpbd::Prediction P,
                                                                   xpbd::HitLists H, int nblocks)
{
    __shared__ int ws[2 * xpbd::kStepWaves];
    if ((int)blockIdx.x >= nblocks) {
        xpbd::scatter_hits(H, blockIdx.x - nblocks, gridDim.x - nblocks, ws);
        return;
    }
    const int i = blockIdx.x * xpbd::kStepBlock + threadIdx.x;
    if (i == 0) step_save[0] = step[0];
    if (i >= nv) return;
    const size_t n = (size_t)nv;
    save[2 * (size_t)i] = pos[2 * (size_t)i];
    save[2 * (size_t)i + 1] = pos[2 * (size_t)i + 1];
    save[2 * n + i] = lo[i];
    save[3 * n + i] = vel[i];
    const float4 d = xpbd::predicted(P, i);
    pos[2 * (size_t)i + 1] = d;
    pred[i] = d;
}

// start of the solve moved by the network's correction (free vertices only)
__global__ void k_apply_corr(float4* __restrict__ pos, const float4* __restrict__ vel, const float4* __restrict__ corr,
                             int nv)
{
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i >= nv || vel[i].w != 0.f) return;
    float4 d = pos[2 * (size_t)i + 1];
    const float4 c = corr[i];
    d.x += c.x;
    d.y += c.y;
    d.z += c.z;
    pos[2 * (size_t)i + 1] = d;
}

// solver correction of this step (end of solve minus prediction); 0 at pins
__global__ void k_store_cprev(const float4* __restrict__ pos, const float4* __restrict__ vel,
                              const float4* __restrict__ pred, float4* __restrict__ cprev, int nv)
{
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i >= nv) return;
    const float4 d = pos[2 * (size_t)i + 1], p = pred[i];
    cprev[i] = vel[i].w != 0.f ? make_float4(0.f, 0.f, 0.f, 0.f) : make_float4(d.x - p.x, d.y - p.y, d.z - p.z, 0.f);
}

__global__ void k_zero_delta(float4* __restrict__ pos, int nv)
{
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i < nv) pos[2 * (size_t)i + 1] = make_float4(0.f, 0.f, 0.f, 0.f);
}

}  // namespace

// ---------------------------------------------------------------------------
// network object
// ---------------------------------------------------------------------------
static uint64_t next_mlp_version()
{
    static std::atomic<uint64_t> counter{ 0 };
    return ++counter;
}

struct xpbd_mlp {
    int device = 0;           // device current at creation (weights and stream live there)
    hipStream_t stream = nullptr;
    float* d_p = nullptr;     // FP32 master parameters
    float* d_g = nullptr;     // gradient
    float* d_m = nullptr;     // Adam first moment
    float* d_v = nullptr;     // Adam second moment
    __bf16* d_w1 = nullptr;   // BF16 copies in the fused-inference layout
    __bf16* d_w2 = nullptr;
    __bf16* d_w3 = nullptr;
    float* d_mean = nullptr;
    float* d_istd = nullptr;
    __bf16* d_wt = nullptr;   // BF16 copies in the training products' operand order
    float* d_part = nullptr;  // weight gradients by run of rows, bias gradients
    char* d_rows = nullptr;   // a minibatch's TrainRows
    int cap_rows = 0;
    float scale = 1.f;
    // Identifies the network and its output scale (the scale is a launch
    // argument of the inference, so graphs that captured it go stale when it
    // changes); never reused within the process.
    uint64_t version = 0;
    float h_mean[24] = {}, h_std[24] = {};  // host copies of the scaling (for xpbd_mlp_save)
    bool has_scaling = false;
    int64_t adam_t = 0;
    // rows of a call (rows = capacity)
    int cap = 0, cap_out = 0, cap_train = 0;
    float *d_X = nullptr, *d_T = nullptr;
    int* d_perm = nullptr;
    float4* d_out = nullptr;
    std::string err;
};

namespace {

int merr(xpbd_mlp* m, int code, const std::string& s)
{
    if (m) m->err = s;
    return code;
}

hipError_t pack(xpbd_mlp* m)
{
    hipLaunchKernelGGL(k_pack, dim3(nb(kH * kH)), dim3(256), 0, m->stream, m->d_p, m->d_w1, m->d_w2, m->d_w3);
    return hipGetLastError();
}

template <typename... P>
void release(P*&... p)
{
    ((void)hipFree(p), ...);
    ((p = nullptr), ...);
}

void free_ws(xpbd_mlp* m)
{
    release(m->d_X, m->d_T, m->d_perm, m->d_out);
    m->cap = m->cap_out = m->cap_train = 0;
}

template <typename T>
hipError_t room(T** p, size_t n)
{
    return hipMalloc(reinterpret_cast<void**>(p), n * sizeof(T));
}

// rows of inputs, and of outputs or (train) of targets and of a permutation
hipError_t ensure_ws(xpbd_mlp* m, int rows, bool train)
{
    const size_t r = (size_t)rows;
    int& cap = train ? m->cap_train : m->cap_out;
    if (rows <= m->cap && rows <= cap) return hipSuccess;
    (void)hipStreamSynchronize(m->stream);
    hipError_t e = hipSuccess;
    if (rows > m->cap) {
        release(m->d_X);
        e = room(&m->d_X, r * kIn);
        m->cap = rows;
    }
    if (rows > cap) {
        if (train) {
            release(m->d_T, m->d_perm);
            if (e == hipSuccess) e = room(&m->d_T, r * kOut);
            if (e == hipSuccess) e = room(&m->d_perm, r);
        } else {
            release(m->d_out);
            if (e == hipSuccess) e = room(&m->d_out, r);
        }
        cap = rows;
    }
    if (e != hipSuccess) free_ws(m);
    return e;
}

// Rows of training that a network keeps room for between calls, 112 bytes each.  One epoch
// over more takes far longer than allocating them again.
constexpr int kKeepRows = 1 << 20;

void trim_ws(xpbd_mlp* m)
{
    if (m->cap_train <= kKeepRows) return;
    release(m->d_T, m->d_perm);
    m->cap_train = 0;
    if (m->cap > m->cap_out) {
        release(m->d_X);
        m->cap = m->cap_out = 0;
        release(m->d_out);
    }
}

constexpr size_t kPart2 = (size_t)kRuns2 * kH * kH, kPart13 = (size_t)kMaxRuns * (kH * kIn + kOut * kH);

// what a minibatch of `rows` rows leaves from launch to launch
hipError_t ensure_minibatch(xpbd_mlp* m, int rows, TrainRows* t)
{
    hipError_t e = hipSuccess;
    if (!m->d_wt) {
        e = room(&m->d_wt, 512 * (size_t)kFrags);
        if (e == hipSuccess) e = room(&m->d_part, kPart2 + kPart13 + 2 * kH + kOut);
        if (e == hipSuccess) e = xpbd::launch_fill_zero(m->stream, m->d_wt, sizeof(__bf16) * 512 * kFrags);
        if (e != hipSuccess) release(m->d_wt, m->d_part);
    }
    const int ld = (rows + kTrainRows - 1) / kTrainRows * kTrainRows;
    if (e == hipSuccess && ld > m->cap_rows) {
        (void)hipStreamSynchronize(m->stream);
        release(m->d_rows);
        m->cap_rows = 0;
        e = room(&m->d_rows, TrainRows::bytes(ld));
        if (e == hipSuccess) m->cap_rows = ld;
    }
    if (e == hipSuccess) t->place(m->d_rows, ld);
    return e;
}

void train_pack(xpbd_mlp* m)
{
    hipLaunchKernelGGL(k_train_pack, dim3(nb(kNParams)), dim3(256), 0, m->stream, m->d_p, m->d_wt);
}

// Gradients of `rows` rows of d_X, d_T, from b0 on through the permutation of nall or (nall 0) as they
// lie, up to their runs' sums; then the sums, into d_g or (lr > 0) into the weights.
struct Adam {
    float lr = 0.f, b1 = 0.f, b2 = 0.f, c1 = 0.f, c2 = 0.f, eps = 0.f;
};
void train_step(xpbd_mlp* m, const TrainRows& t, int rows, int b0, int nall, const Adam& a)
{
    const Runs r2 = runs_of(rows, 16), r13 = runs_of(rows, 4);   // tiles of 32 x 32: 128 x 128; 128 x 24 and 3 x 128
    float *part13 = m->d_part + kPart2, *bias = part13 + kPart13;
    hipLaunchKernelGGL(k_train_rows, dim3((rows + kTrainRows - 1) / kTrainRows), dim3(kTrainThreads), 0, m->stream, m->d_X,
                       m->d_T, nall > 0 ? m->d_perm : nullptr, b0, nall, rows, m->d_mean, m->d_istd, 1.0f / m->scale,
                       m->d_p, m->d_wt, t);
    hipLaunchKernelGGL(k_train_weights, dim3(4 * r2.n + r13.n + 2 * kH + kOut), dim3(256), 0, m->stream, t, rows, r2, r13,
                       m->d_part, part13, bias);
    if (a.lr > 0.f)
        hipLaunchKernelGGL(k_train_update<true>, dim3(nb(kNParams)), dim3(256), 0, m->stream, m->d_part, r2.n, part13,
                           r13.n, bias, nullptr, m->d_p, m->d_m, m->d_v, m->d_wt, a.lr, a.b1, a.b2, a.c1, a.c2, a.eps);
    else
        hipLaunchKernelGGL(k_train_update<false>, dim3(nb(kNParams)), dim3(256), 0, m->stream, m->d_part, r2.n, part13,
                           r13.n, bias, m->d_g, nullptr, nullptr, nullptr, nullptr, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f);
}

double read_loss(xpbd_mlp* m, const TrainRows& t, int rows)
{
    std::vector<double> lp((rows + kTrainRows - 1) / kTrainRows);
    (void)hipMemcpyAsync(lp.data(), t.loss, sizeof(double) * lp.size(), hipMemcpyDeviceToHost, m->stream);
    (void)hipStreamSynchronize(m->stream);
    double s = 0;
    for (double v : lp) s += v;
    return s / ((double)rows * kOut);
}

}  // namespace

extern "C" int xpbd_mlp_num_params(int32_t* out)
{
    if (!out) return XPBD_E_INVALID_ARG;
    *out = kNParams;
    return XPBD_OK;
}

extern "C" int xpbd_mlp_create(xpbd_mlp** out)
{
    if (!out) return XPBD_E_INVALID_ARG;
    *out = nullptr;
    xpbd_mlp* m = new (std::nothrow) xpbd_mlp();
    if (!m) return XPBD_E_NOMEM;
    m->version = next_mlp_version();
    hipError_t e = hipGetDevice(&m->device);
    if (e == hipSuccess) e = hipStreamCreateWithFlags(&m->stream, hipStreamNonBlocking);
    auto A = [&](void** p, size_t bytes) {
        if (e == hipSuccess) e = hipMalloc(p, bytes);
    };
    A(reinterpret_cast<void**>(&m->d_p), sizeof(float) * kNParams);
    A(reinterpret_cast<void**>(&m->d_g), sizeof(float) * kNParams);
    A(reinterpret_cast<void**>(&m->d_m), sizeof(float) * kNParams);
    A(reinterpret_cast<void**>(&m->d_v), sizeof(float) * kNParams);
    A(reinterpret_cast<void**>(&m->d_w1), sizeof(__bf16) * kH * kInP);
    A(reinterpret_cast<void**>(&m->d_w2), sizeof(__bf16) * kH * kH);
    A(reinterpret_cast<void**>(&m->d_w3), sizeof(__bf16) * kOutP * kH);
    A(reinterpret_cast<void**>(&m->d_mean), sizeof(float) * kIn);
    A(reinterpret_cast<void**>(&m->d_istd), sizeof(float) * kIn);
    if (e != hipSuccess) {
        xpbd_mlp_destroy(m);
        return XPBD_E_NOMEM;
    }
    // Glorot-uniform initial weights, zero biases (fixed seed), identity scaling
    std::vector<float> p(kNParams, 0.f);
    std::mt19937 rng(20099u);
    auto init = [&](int off, int fan_out, int fan_in) {
        const float a = std::sqrt(6.0f / (float)(fan_in + fan_out));
        std::uniform_real_distribution<float> U(-a, a);
        for (int i = 0; i < fan_out * fan_in; i++) p[off + i] = U(rng);
    };
    init(oW1, kH, kIn);
    init(oW2, kH, kH);
    init(oW3, kOut, kH);
    std::vector<float> zero(kNParams, 0.f), mean(kIn, 0.f), one(kIn, 1.f);
    e = hipMemcpy(m->d_p, p.data(), sizeof(float) * kNParams, hipMemcpyHostToDevice);
    if (e == hipSuccess) e = hipMemcpy(m->d_m, zero.data(), sizeof(float) * kNParams, hipMemcpyHostToDevice);
    if (e == hipSuccess) e = hipMemcpy(m->d_v, zero.data(), sizeof(float) * kNParams, hipMemcpyHostToDevice);
    if (e == hipSuccess) e = hipMemcpy(m->d_g, zero.data(), sizeof(float) * kNParams, hipMemcpyHostToDevice);
    if (e == hipSuccess) e = hipMemcpy(m->d_mean, mean.data(), sizeof(float) * kIn, hipMemcpyHostToDevice);
    if (e == hipSuccess) e = hipMemcpy(m->d_istd, one.data(), sizeof(float) * kIn, hipMemcpyHostToDevice);
    if (e == hipSuccess) e = pack(m);
    if (e == hipSuccess) e = hipStreamSynchronize(m->stream);
    if (e != hipSuccess) {
        xpbd_mlp_destroy(m);
        return XPBD_E_HIP;
    }
    *out = m;
    return XPBD_OK;
}

extern "C" int xpbd_mlp_destroy(xpbd_mlp* m)
{
    if (!m) return XPBD_OK;
    if (m->stream) (void)hipStreamSynchronize(m->stream);
    free_ws(m);
    release(m->d_p, m->d_g, m->d_m, m->d_v, m->d_w1, m->d_w2, m->d_w3, m->d_mean, m->d_istd, m->d_wt, m->d_part,
            m->d_rows);
    if (m->stream) (void)hipStreamDestroy(m->stream);
    delete m;
    return XPBD_OK;
}

extern "C" const char* xpbd_mlp_last_error(const xpbd_mlp* m) { return m ? m->err.c_str() : "null network"; }

extern "C" int xpbd_mlp_set_params(xpbd_mlp* m, const float* params)
{
    if (!m || !params) return XPBD_E_INVALID_ARG;
    for (int i = 0; i < kNParams; i++)
        if (!std::isfinite(params[i])) return merr(m, XPBD_E_NONFINITE, "non-finite parameter");
    hipError_t e = hipMemcpyAsync(m->d_p, params, sizeof(float) * kNParams, hipMemcpyHostToDevice, m->stream);
    if (e == hipSuccess) e = pack(m);
    if (e == hipSuccess) e = hipStreamSynchronize(m->stream);
    return e == hipSuccess ? XPBD_OK : merr(m, XPBD_E_HIP, hipGetErrorString(e));
}

extern "C" int xpbd_mlp_get_params(xpbd_mlp* m, float* params)
{
    if (!m || !params) return XPBD_E_INVALID_ARG;
    hipError_t e = hipMemcpyAsync(params, m->d_p, sizeof(float) * kNParams, hipMemcpyDeviceToHost, m->stream);
    if (e == hipSuccess) e = hipStreamSynchronize(m->stream);
    return e == hipSuccess ? XPBD_OK : merr(m, XPBD_E_HIP, hipGetErrorString(e));
}

extern "C" int xpbd_mlp_set_scaling(xpbd_mlp* m, const float* mean_in, const float* std_in, float scale_out)
{
    if (!m || !mean_in || !std_in || !(scale_out > 0) || !std::isfinite(scale_out)) return XPBD_E_INVALID_ARG;
    float istd[kIn];
    for (int k = 0; k < kIn; k++) {
        if (!(std_in[k] > 0) || !std::isfinite(std_in[k]) || !std::isfinite(mean_in[k]))
            return merr(m, XPBD_E_INVALID_ARG, "std must be positive and finite");
        istd[k] = 1.0f / std_in[k];
    }
    hipError_t e = hipMemcpyAsync(m->d_mean, mean_in, sizeof(float) * kIn, hipMemcpyHostToDevice, m->stream);
    if (e == hipSuccess) e = hipMemcpyAsync(m->d_istd, istd, sizeof(float) * kIn, hipMemcpyHostToDevice, m->stream);
    if (e == hipSuccess) e = hipStreamSynchronize(m->stream);
    m->scale = scale_out;
    m->version = next_mlp_version();
    if (e == hipSuccess) {
        std::memcpy(m->h_mean, mean_in, sizeof(float) * kIn);
        std::memcpy(m->h_std, std_in, sizeof(float) * kIn);
        m->has_scaling = true;
    }
    return e == hipSuccess ? XPBD_OK : merr(m, XPBD_E_HIP, hipGetErrorString(e));
}

namespace {
constexpr char kMlpMagic[8] = { 'X', 'P', 'B', 'D', 'M', 'L', 'P', '1' };
}

extern "C" int xpbd_mlp_save(xpbd_mlp* m, const char* path)
{
    if (!m || !path) return XPBD_E_INVALID_ARG;
    if (!m->has_scaling) return merr(m, XPBD_E_INVALID_ARG, "no feature scaling set");
    std::vector<float> p(kNParams);
    int rc = xpbd_mlp_get_params(m, p.data());
    if (rc) return rc;
    FILE* f = std::fopen(path, "wb");
    if (!f) return merr(m, XPBD_E_INVALID_ARG, std::string("cannot write ") + path);
    const int32_t sizes[2] = { kNParams, kIn };
    bool ok = std::fwrite(kMlpMagic, 1, sizeof(kMlpMagic), f) == sizeof(kMlpMagic) &&
              std::fwrite(sizes, sizeof(int32_t), 2, f) == 2 &&
              std::fwrite(p.data(), sizeof(float), kNParams, f) == (size_t)kNParams &&
              std::fwrite(m->h_mean, sizeof(float), kIn, f) == (size_t)kIn &&
              std::fwrite(m->h_std, sizeof(float), kIn, f) == (size_t)kIn &&
              std::fwrite(&m->scale, sizeof(float), 1, f) == 1;
    ok = (std::fclose(f) == 0) && ok;
    return ok ? XPBD_OK : merr(m, XPBD_E_INVALID_ARG, std::string("short write to ") + path);
}

extern "C" int xpbd_mlp_load(xpbd_mlp* m, const char* path)
{
    if (!m || !path) return XPBD_E_INVALID_ARG;
    FILE* f = std::fopen(path, "rb");
    if (!f) return merr(m, XPBD_E_INVALID_ARG, std::string("cannot read ") + path);
    char magic[8];
    int32_t sizes[2];
    std::vector<float> p(kNParams);
    float mean[kIn], sd[kIn], scale = 0.f;
    bool ok = std::fread(magic, 1, sizeof(magic), f) == sizeof(magic) &&
              std::memcmp(magic, kMlpMagic, sizeof(magic)) == 0 && std::fread(sizes, sizeof(int32_t), 2, f) == 2 &&
              sizes[0] == kNParams && sizes[1] == kIn &&
              std::fread(p.data(), sizeof(float), kNParams, f) == (size_t)kNParams &&
              std::fread(mean, sizeof(float), kIn, f) == (size_t)kIn &&
              std::fread(sd, sizeof(float), kIn, f) == (size_t)kIn && std::fread(&scale, sizeof(float), 1, f) == 1;
    char extra;
    ok = ok && std::fread(&extra, 1, 1, f) == 0;  // nothing after the scale
    std::fclose(f);
    if (!ok) return merr(m, XPBD_E_INVALID_ARG, std::string("not a network file of this layout: ") + path);
    int rc = xpbd_mlp_set_params(m, p.data());
    return rc ? rc : xpbd_mlp_set_scaling(m, mean, sd, scale);
}

namespace {
// fused inference on device rows: out[r] = scale * MLP(standardised X[r])
hipError_t mlp_infer(xpbd_mlp* m, hipStream_t s, const float* dX, int n, float4* dout)
{
    if (n <= 0) return hipSuccess;
    const int tiles = (n + kFwdRows - 1) / kFwdRows;
    const int grid = tiles < 512 ? tiles : 512;
    hipLaunchKernelGGL(k_mlp_fused, dim3(grid), dim3(256), 0, s, dX, n, m->d_w1, m->d_w2, m->d_w3, m->d_p, m->d_mean,
                       m->d_istd, m->scale, dout, nullptr);
    return hipGetLastError();
}
}  // namespace

// Rows from which the outputs are packed on the device: a launch is 5 us (1 row: 34 us
// against 29), the host's loop and its fresh pages 0.5 us a thousand rows (10,000 rows:
// 75 both ways, 185,193: 669 against 755).
constexpr int kPackRows = 16384;

extern "C" int xpbd_mlp_forward(xpbd_mlp* m, int32_t n, const float* x, float* out)
{
    if (!m || n < 0 || (n > 0 && (!x || !out))) return XPBD_E_INVALID_ARG;
    if (n == 0) return XPBD_OK;
    hipError_t e = ensure_ws(m, n, false);
    if (e != hipSuccess) return merr(m, XPBD_E_NOMEM, hipGetErrorString(e));
    e = hipMemcpyAsync(m->d_X, x, sizeof(float) * kIn * (size_t)n, hipMemcpyHostToDevice, m->stream);
    if (e == hipSuccess) e = mlp_infer(m, m->stream, m->d_X, n, m->d_out);
    if (n < kPackRows) {
        std::vector<float4> o(n);
        if (e == hipSuccess)
            e = hipMemcpyAsync(o.data(), m->d_out, sizeof(float4) * (size_t)n, hipMemcpyDeviceToHost, m->stream);
        if (e == hipSuccess) e = hipStreamSynchronize(m->stream);
        if (e != hipSuccess) return merr(m, XPBD_E_HIP, hipGetErrorString(e));
        for (int i = 0; i < n; i++) {
            out[3 * (size_t)i] = o[i].x;
            out[3 * (size_t)i + 1] = o[i].y;
            out[3 * (size_t)i + 2] = o[i].z;
        }
        return XPBD_OK;
    }
    // the rows' buffer is free again: packed there, as the caller gets them
    if (e == hipSuccess) {
        hipLaunchKernelGGL(k_pack3, dim3(nb(n)), dim3(256), 0, m->stream, m->d_out, n, m->d_X);
        e = hipGetLastError();
    }
    if (e == hipSuccess)
        e = hipMemcpyAsync(out, m->d_X, sizeof(float) * kOut * (size_t)n, hipMemcpyDeviceToHost, m->stream);
    if (e == hipSuccess) e = hipStreamSynchronize(m->stream);
    return e == hipSuccess ? XPBD_OK : merr(m, XPBD_E_HIP, hipGetErrorString(e));
}

// ---------------------------------------------------------------------------
// Forward without allocation: the rows are staged through a fixed file-scope
// device array instead of the network's workspace (which xpbd_mlp_forward grows
// with hipMalloc).  Each GPU holds its own copy of the array; its address on a
// device is looked up once (hipGetSymbolAddress with that device current) and
// kept, since the array's name in host code is not a device address.
// ---------------------------------------------------------------------------
namespace {
constexpr int kNoAllocRows = XPBD_MLP_NOALLOC_MAX_ROWS;
// per row: 24 input floats, a float4 network output, 3 packed output floats
constexpr size_t kScratchFloats = (size_t)kNoAllocRows * (kIn + 4 + kOut);
static __device__ __align__(256) float scratch[kScratchFloats];

constexpr int kMaxDevices = 64;
std::mutex g_scratch_mutex;
float* g_scratch_ptr[kMaxDevices] = {};

// The calling thread's device is made `device` for the lookup and restored.
hipError_t scratch_on(int device, float** out)
{
    if (device < 0 || device >= kMaxDevices) return hipErrorInvalidDevice;
    std::lock_guard<std::mutex> lock(g_scratch_mutex);
    if (!g_scratch_ptr[device]) {
        int cur = 0;
        hipError_t e = hipGetDevice(&cur);
        if (e == hipSuccess && cur != device) e = hipSetDevice(device);
        void* p = nullptr;
        if (e == hipSuccess) e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (cur != device) (void)hipSetDevice(cur);
        if (e != hipSuccess) return e;
        g_scratch_ptr[device] = static_cast<float*>(p);
    }
    *out = g_scratch_ptr[device];
    return hipSuccess;
}

}  // namespace

extern "C" int xpbd_mlp_forward_noalloc(xpbd_mlp* m, int32_t n, const float* x, float* out)
{
    if (!m || n < 0 || (n > 0 && (!x || !out))) return XPBD_E_INVALID_ARG;
    if (n > kNoAllocRows)
        return merr(m, XPBD_E_INVALID_ARG,
                    "xpbd_mlp_forward_noalloc: " + std::to_string(n) + " rows exceed the fixed scratch of " +
                        std::to_string(kNoAllocRows) + " rows (call it in chunks, or use xpbd_mlp_forward)");
    if (n == 0) return XPBD_OK;
    float* base = nullptr;
    hipError_t e = scratch_on(m->device, &base);
    if (e != hipSuccess) return merr(m, XPBD_E_HIP, std::string("scratch lookup: ") + hipGetErrorString(e));
    float* dX = base;                                                                   // n x 24
    float4* d4 = reinterpret_cast<float4*>(base + (size_t)kNoAllocRows * kIn);         // n float4
    float* d3 = base + (size_t)kNoAllocRows * (kIn + 4);                                // n x 3
    e = hipMemcpyAsync(dX, x, sizeof(float) * kIn * (size_t)n, hipMemcpyHostToDevice, m->stream);
    if (e == hipSuccess) e = mlp_infer(m, m->stream, dX, n, d4);
    if (e == hipSuccess) {
        hipLaunchKernelGGL(k_pack3, dim3(nb(n)), dim3(256), 0, m->stream, d4, n, d3);
        e = hipGetLastError();
    }
    if (e == hipSuccess) e = hipMemcpyAsync(out, d3, sizeof(float) * kOut * (size_t)n, hipMemcpyDeviceToHost, m->stream);
    if (e == hipSuccess) e = hipStreamSynchronize(m->stream);
    return e == hipSuccess ? XPBD_OK : merr(m, XPBD_E_HIP, hipGetErrorString(e));
}

extern "C" int xpbd_mlp_loss_grad(xpbd_mlp* m, int32_t n, const float* x, const float* y, double* loss, float* grad)
{
    if (!m || n <= 0 || !x || !y || !loss) return XPBD_E_INVALID_ARG;
    hipError_t e = ensure_ws(m, n, true);
    TrainRows t;
    if (e == hipSuccess) e = ensure_minibatch(m, n, &t);
    if (e != hipSuccess) return merr(m, XPBD_E_NOMEM, hipGetErrorString(e));
    e = hipMemcpyAsync(m->d_X, x, sizeof(float) * kIn * (size_t)n, hipMemcpyHostToDevice, m->stream);
    if (e == hipSuccess)
        e = hipMemcpyAsync(m->d_T, y, sizeof(float) * kOut * (size_t)n, hipMemcpyHostToDevice, m->stream);
    if (e != hipSuccess) return merr(m, XPBD_E_HIP, hipGetErrorString(e));
    train_pack(m);
    train_step(m, t, n, 0, 0, Adam{});
    e = hipGetLastError();
    if (e != hipSuccess) return merr(m, XPBD_E_HIP, hipGetErrorString(e));
    *loss = read_loss(m, t, n);
    if (grad) {
        e = hipMemcpyAsync(grad, m->d_g, sizeof(float) * kNParams, hipMemcpyDeviceToHost, m->stream);
        if (e == hipSuccess) e = hipStreamSynchronize(m->stream);
    }
    return e == hipSuccess ? XPBD_OK : merr(m, XPBD_E_HIP, hipGetErrorString(e));
}

extern "C" int xpbd_mlp_train(xpbd_mlp* m, int32_t n, const float* x, const float* y, int32_t batch, int32_t epochs,
                              float lr, uint64_t seed, double* final_loss)
{
    if (!m || n <= 0 || !x || !y || batch <= 0 || epochs < 0 || !(lr > 0) || !std::isfinite(lr))
        return XPBD_E_INVALID_ARG;
    if (batch > n) batch = n;
    // all samples live on the device; each epoch takes its minibatches through a
    // seeded permutation
    hipError_t e = ensure_ws(m, n, true);
    TrainRows t;
    if (e == hipSuccess) e = ensure_minibatch(m, batch, &t);
    if (e != hipSuccess) return merr(m, XPBD_E_NOMEM, hipGetErrorString(e));
    e = hipMemcpyAsync(m->d_X, x, sizeof(float) * kIn * (size_t)n, hipMemcpyHostToDevice, m->stream);
    if (e == hipSuccess)
        e = hipMemcpyAsync(m->d_T, y, sizeof(float) * kOut * (size_t)n, hipMemcpyHostToDevice, m->stream);
    if (e != hipSuccess) {
        (void)hipStreamSynchronize(m->stream);
        return merr(m, XPBD_E_NOMEM, hipGetErrorString(e));
    }
    train_pack(m);
    std::mt19937_64 rng(seed);
    std::vector<int32_t> perm(n);
    for (int i = 0; i < n; i++) perm[i] = i;
    const float b1 = 0.9f, b2 = 0.999f, eps = 1e-8f;
    double last = 0;
    const int nbatch = n / batch > 0 ? n / batch : 1;
    for (int ep = 0; ep < epochs && e == hipSuccess; ep++) {
        std::shuffle(perm.begin(), perm.end(), rng);
        e = hipMemcpyAsync(m->d_perm, perm.data(), sizeof(int) * (size_t)n, hipMemcpyHostToDevice, m->stream);
        for (int bi = 0; bi < nbatch && e == hipSuccess; bi++) {
            m->adam_t++;
            const float c1 = 1.f - std::pow(b1, (float)m->adam_t), c2 = 1.f - std::pow(b2, (float)m->adam_t);
            train_step(m, t, batch, bi * batch, n, Adam{ lr, b1, b2, c1, c2, eps });
            e = hipGetLastError();
        }
        // the host permutation is rewritten next epoch: wait for its copy
        if (e == hipSuccess) last = read_loss(m, t, batch);
    }
    if (e == hipSuccess) e = pack(m);
    if (e == hipSuccess) e = hipStreamSynchronize(m->stream);
    (void)hipStreamSynchronize(m->stream);
    trim_ws(m);
    if (final_loss) *final_loss = last;
    return e == hipSuccess ? XPBD_OK : merr(m, XPBD_E_HIP, hipGetErrorString(e));
}

// ---------------------------------------------------------------------------
// learned step on a solver handle
// ---------------------------------------------------------------------------
namespace xpbd {

struct Learned {
    xpbd_mlp* mlp = nullptr;
    int nv = 0;
    int* d_nb_off = nullptr;
    int* d_nb = nullptr;
    float2* d_vmat = nullptr;
    float* d_pinfrac = nullptr;
    float* d_feat = nullptr;     // nv x 24
    float4* d_pred = nullptr;    // in-step motion after the prediction
    float4* d_cprev = nullptr;   // previous step's solver correction
    float4* d_corr = nullptr;    // network output
    float4* d_save = nullptr;    // snapshot for the fallback: pos (2 nv), lo (nv), vel (nv)
    unsigned long long* d_step_save = nullptr;
    double* d_res = nullptr;     // squared residual of the learned solve
    // Captured learned steps, one per (network version, handle graph
    // generation, detection, iterations, start mode).
    struct Graph {
        uint64_t net = 0, gen = 0;
        int det = 0, iters = 0, start = 0;
        hipGraphExec_t exec = nullptr;
    };
    std::vector<Graph> graphs;
    // inference timing (kernel timing mode of the handle)
    hipEvent_t ev0 = nullptr, ev1 = nullptr;
    double mlp_ms = 0;
    int64_t mlp_calls = 0;
    int64_t steps = 0, fallbacks = 0;
    // XPBD_LEARNED_START_*: how the solve after the network's correction starts
    int start = XPBD_LEARNED_START_MULTIPLIERS;
};

static void free_learned(Learned* L)
{
    if (!L) return;
    for (auto& g : L->graphs)
        if (g.exec) (void)hipGraphExecDestroy(g.exec);
    void* bufs[] = { L->d_nb_off, L->d_nb, L->d_vmat, L->d_pinfrac, L->d_feat, L->d_pred,
                     L->d_cprev,  L->d_corr, L->d_save, L->d_step_save, L->d_res };
    for (void* b : bufs)
        if (b) (void)hipFree(b);
    if (L->ev0) (void)hipEventDestroy(L->ev0);
    if (L->ev1) (void)hipEventDestroy(L->ev1);
    delete L;
}

void destroy_learned(xpbd_handle* h)
{
    if (!h || !h->learned) return;
    (void)hipStreamSynchronize(h->stream);
    free_learned(h->learned);
    h->learned = nullptr;
}

int learned_reset_history(xpbd_handle* h)
{
    if (!h->learned) return XPBD_OK;
    hipError_t e = launch_fill_zero(h->stream, h->learned->d_cprev, sizeof(float4) * (size_t)h->nv);
    if (e == hipSuccess) e = hipStreamSynchronize(h->stream);
    return e == hipSuccess ? XPBD_OK : hip_err(h, e, "learned history reset");
}

// Device buffers of the learned step (1-ring CSR, material summary, scratch).
static int ensure_learned(xpbd_handle* h)
{
    if (h->learned) return XPBD_OK;
    const int nv = h->nv, nt = h->nt;
    // 1-ring neighbours from the element list (sorted, unique)
    std::vector<int64_t> pairs;
    pairs.reserve(12 * (size_t)nt);
    for (int e = 0; e < nt; e++) {
        const int32_t* t = &h->tets_host[4 * (size_t)e];
        for (int a = 0; a < 4; a++)
            for (int b = 0; b < 4; b++)
                if (a != b) pairs.push_back(((int64_t)t[a] << 32) | (uint32_t)t[b]);
    }
    std::sort(pairs.begin(), pairs.end());
    pairs.erase(std::unique(pairs.begin(), pairs.end()), pairs.end());
    std::vector<int32_t> off(nv + 1, 0), nbr(pairs.size());
    for (size_t k = 0; k < pairs.size(); k++) {
        off[(pairs[k] >> 32) + 1]++;
        nbr[k] = (int32_t)(pairs[k] & 0xffffffff);
    }
    for (int v = 0; v < nv; v++) off[v + 1] += off[v];
    std::vector<float> pinfrac(nv, 0.f);
    for (int v = 0; v < nv; v++) {
        int c = 0;
        for (int k = off[v]; k < off[v + 1]; k++) c += h->pinned[nbr[k]] ? 1 : 0;
        pinfrac[v] = off[v + 1] > off[v] ? (float)c / (float)(off[v + 1] - off[v]) : 0.f;
    }
    Learned* L = new (std::nothrow) Learned();
    if (!L) return set_err(h, XPBD_E_NOMEM, "learned state allocation failed");
    L->nv = nv;
    hipError_t e = hipSuccess;
    auto A = [&](auto** p, size_t bytes) {
        if (e == hipSuccess) e = hipMalloc(reinterpret_cast<void**>(p), bytes > 0 ? bytes : 16);
    };
    A(&L->d_nb_off, sizeof(int) * (nv + 1));
    A(&L->d_nb, sizeof(int) * nbr.size());
    A(&L->d_vmat, sizeof(float2) * nv);
    A(&L->d_pinfrac, sizeof(float) * nv);
    A(&L->d_feat, sizeof(float) * kIn * (size_t)nv);
    A(&L->d_pred, sizeof(float4) * nv);
    A(&L->d_cprev, sizeof(float4) * nv);
    A(&L->d_corr, sizeof(float4) * nv);
    A(&L->d_save, sizeof(float4) * 4 * (size_t)nv);
    A(&L->d_step_save, sizeof(unsigned long long));
    A(&L->d_res, sizeof(double));
    if (e == hipSuccess) e = hipMemcpy(L->d_nb_off, off.data(), sizeof(int) * (nv + 1), hipMemcpyHostToDevice);
    if (e == hipSuccess && !nbr.empty())
        e = hipMemcpy(L->d_nb, nbr.data(), sizeof(int) * nbr.size(), hipMemcpyHostToDevice);
    if (e == hipSuccess) e = hipMemcpy(L->d_vmat, h->vmat.data(), sizeof(float2) * nv, hipMemcpyHostToDevice);
    if (e == hipSuccess) e = hipMemcpy(L->d_pinfrac, pinfrac.data(), sizeof(float) * nv, hipMemcpyHostToDevice);
    if (e == hipSuccess) e = hipEventCreate(&L->ev0);
    if (e == hipSuccess) e = hipEventCreate(&L->ev1);
    if (e == hipSuccess) e = launch_fill_zero(h->stream, L->d_cprev, sizeof(float4) * nv);
    if (e == hipSuccess) e = hipStreamSynchronize(h->stream);
    if (e != hipSuccess) {
        free_learned(L);
        return hip_err(h, e, "learned set-up");
    }
    h->learned = L;
    return XPBD_OK;
}

static int enqueue_features(xpbd_handle* h)
{
    Learned* L = h->learned;
    hipLaunchKernelGGL(k_features, dim3(nb(h->nv)), dim3(256), 0, h->stream, h->d_pos, h->d_vel, L->d_cprev,
                       L->d_nb_off, L->d_nb, L->d_vmat, L->d_pinfrac, h->nv, L->d_feat);
    hipError_t e = hipGetLastError();
    return e == hipSuccess ? XPBD_OK : hip_err(h, e, "features launch");
}

static int enqueue_copy_pred(xpbd_handle* h)
{
    hipLaunchKernelGGL(k_copy_delta, dim3(nb(h->nv)), dim3(256), 0, h->stream, h->d_pos, h->learned->d_pred, h->nv);
    hipError_t e = hipGetLastError();
    return e == hipSuccess ? XPBD_OK : hip_err(h, e, "copy launch");
}

static int enqueue_store_cprev(xpbd_handle* h)
{
    Learned* L = h->learned;
    hipLaunchKernelGGL(k_store_cprev, dim3(nb(h->nv)), dim3(256), 0, h->stream, h->d_pos, h->d_vel, L->d_pred,
                       L->d_cprev, h->nv);
    hipError_t e = hipGetLastError();
    return e == hipSuccess ? XPBD_OK : hip_err(h, e, "correction launch");
}

// Multiplier start of the learned step, on the corrected positions: the
// contacts are projected once from zero multipliers (a Gauss-Seidel contact
// pass, or the Jacobi contact sum), so that the start does not penetrate the
// collider, then every element's multipliers are set to -C / alpha~ there.
// Attachment multipliers start at zero.  The iterations that follow keep all
// of them.
static int enqueue_multiplier_start(xpbd_handle* h)
{
    hipStream_t s = h->stream;
    hipError_t e = hipSuccess;
    if (h->natt > 0) e = launch_fill_zero(s, h->d_att_lam, sizeof(double) * (size_t)h->natt);
    if (e == hipSuccess && contacts_enabled(h)) {
        if (h->params.solver == XPBD_SOLVER_GS_COLORED) {
            e = launch_contacts_gs(s, h->d_faces, h->d_fci_off, h->nfcolors, h->ninst, h->d_cpos, h->d_clist,
                                   h->d_rest, h->d_pos, h->d_lo, h->d_cp, h->d_cn, h->d_cb, h->d_clam, true);
        } else {
            int rc = enqueue_contacts_jacobi(h, true);
            if (rc) return rc;
            e = launch_jacobi_apply(s, h->d_pos, h->d_acc, h->nv);
        }
    }
    if (e == hipSuccess) e = launch_lambda_start(s, tet_arrays(h), h->d_pos, h->d_lo, h->nt);
    return e == hipSuccess ? XPBD_OK : hip_err(h, e, "multiplier start");
}

// Consistent start (XPBD_LEARNED_START_CONSISTENT, the oracle's orc_step_learned):
// the multipliers lambda0 = -C / alpha~ at the corrected positions xl = xt + corr,
// then the positions x0 = xt + M^-1 sum grad C(xl)^T lambda0 from the kept
// prediction, so that the momentum balance M (x - xt) = grad C^T lambda, which
// the XPBD updates preserve, holds at the first iteration.  Contact and
// attachment multipliers start at zero, as in a plain solve.
static int enqueue_consistent_start(xpbd_handle* h)
{
    hipStream_t s = h->stream;
    hipError_t e = hipSuccess;
    if (h->natt > 0) e = launch_fill_zero(s, h->d_att_lam, sizeof(double) * (size_t)h->natt);
    if (e == hipSuccess && h->nf > 0) e = launch_fill_zero(s, h->d_clam, sizeof(double) * (size_t)h->nf);
    const TetArrays ta = tet_arrays(h);
    if (e == hipSuccess) e = launch_lambda_start(s, ta, h->d_pos, h->d_lo, h->nt);
    if (e == hipSuccess) e = launch_element_forces(s, ta, element_force_args(h));
    if (e == hipSuccess) e = launch_consistent_shift(s, h->d_pos, h->learned->d_pred, h->d_vt_off, h->d_eforce, h->nv);
    return e == hipSuccess ? XPBD_OK : hip_err(h, e, "consistent start");
}

}  // namespace xpbd

using namespace xpbd;

extern "C" int xpbd_attach_mlp(xpbd_handle* h, xpbd_mlp* m)
{
    if (!h) return XPBD_E_INVALID_ARG;
    if (!m) {
        if (h->learned) h->learned->mlp = nullptr;
        return XPBD_OK;
    }
    int rc = ensure_learned(h);
    if (rc) return rc;
    h->learned->mlp = m;
    return XPBD_OK;
}

extern "C" int xpbd_features(xpbd_handle* h, float* out)
{
    if (!h || !out) return h ? set_err(h, XPBD_E_INVALID_ARG, "out is NULL") : XPBD_E_INVALID_ARG;
    int rc = ensure_learned(h);
    if (rc) return rc;
    // features of the state after this step's prediction; the prediction is undone afterwards
    if ((rc = enqueue_predict(h)) || (rc = enqueue_features(h))) return rc;
    hipLaunchKernelGGL(k_zero_delta, dim3(nb(h->nv)), dim3(256), 0, h->stream, h->d_pos, h->nv);
    hipError_t e = hipGetLastError();
    if (e == hipSuccess)
        e = hipMemcpyAsync(out, h->learned->d_feat, sizeof(float) * kIn * (size_t)h->nv, hipMemcpyDeviceToHost,
                           h->stream);
    if (e == hipSuccess) e = hipStreamSynchronize(h->stream);
    return e == hipSuccess ? XPBD_OK : hip_err(h, e, "features");
}

extern "C" int xpbd_collect_training(xpbd_handle* h, int32_t nsteps, int32_t cap, float* x, float* y, int32_t* rows)
{
    if (!h || nsteps < 0 || cap < 0 || !rows || (cap > 0 && (!x || !y)))
        return h ? set_err(h, XPBD_E_INVALID_ARG, "collect_training: bad arguments") : XPBD_E_INVALID_ARG;
    int rc = ensure_learned(h);
    if (rc) return rc;
    Learned* L = h->learned;
    const int nv = h->nv;
    std::vector<float> feat((size_t)kIn * nv);
    std::vector<float4> corr(nv);
    int32_t count = 0;
    for (int32_t s = 0; s < nsteps; s++) {
        const bool det = detect_this_step(h);
        if (det && (rc = enqueue_detect(h))) return rc;
        if ((rc = enqueue_predict(h)) || (rc = enqueue_copy_pred(h)) || (rc = enqueue_features(h))) return rc;
        hipError_t e = hipMemcpyAsync(feat.data(), L->d_feat, sizeof(float) * feat.size(), hipMemcpyDeviceToHost,
                                      h->stream);
        if (e != hipSuccess) return hip_err(h, e, "collect features");
        if ((rc = enqueue_iterations(h, h->params.iters, false))) return rc;
        if (records_residuals(h) && (rc = enqueue_step_residual(h))) return rc;
        if ((rc = enqueue_local_collision(h))) return rc;
        if ((rc = enqueue_store_cprev(h)) || (rc = enqueue_finish(h))) return rc;
        e = hipMemcpyAsync(corr.data(), L->d_cprev, sizeof(float4) * nv, hipMemcpyDeviceToHost, h->stream);
        if (e == hipSuccess) e = hipStreamSynchronize(h->stream);
        if (e != hipSuccess) return hip_err(h, e, "collect targets");
        h->host_step++;
        for (int i = 0; i < nv && count < cap; i++) {
            if (h->pinned[i]) continue;
            std::memcpy(x + (size_t)count * kIn, &feat[(size_t)i * kIn], sizeof(float) * kIn);
            y[(size_t)count * kOut] = corr[i].x;
            y[(size_t)count * kOut + 1] = corr[i].y;
            y[(size_t)count * kOut + 2] = corr[i].z;
            count++;
        }
    }
    *rows = count;
    return XPBD_OK;
}

namespace xpbd {
// The learned step up to its end, before the fallback decision: detection (on
// the plain solver's cadence), a snapshot of the start-of-step state, the
// prediction, features, network correction, the multiplier start, iters
// iterations, the squared residual into L->d_res, then the rest of the step
// (EVERY_SUBSTEP residual, local collision passes, the correction history and
// the velocity update).  A fallback restores the snapshot and redoes the
// whole step as the plain solver does, so finishing the step before the
// decision changes nothing on either branch.
static int enqueue_learned_attempt(xpbd_handle* h, int32_t iters, bool det, bool timed)
{
    Learned* L = h->learned;
    const int nv = h->nv;
    hipStream_t s = h->stream;
    int rc;
    det = det && h->nf > 0;
    if (det && (rc = enqueue_flags(h))) return rc;
    const HitLists H = det ? hit_lists(h) : HitLists{};
    hipLaunchKernelGGL(k_learned_begin, dim3(nb(nv) + (det ? compact_blocks(h->nf) : 0)), dim3(kStepBlock), 0, s, h->d_pos,
                       h->d_lo, h->d_vel, nv, h->d_step, L->d_save, L->d_step_save, L->d_pred, prediction(h), H,
                       (int)nb(nv));
    hipError_t e = hipGetLastError();
    if (e == hipSuccess && h->primary_residual) e = launch_keep_prediction(s, h->d_pos, h->d_pred, nv);
    if (e != hipSuccess) return hip_err(h, e, "learned start");
    if ((rc = enqueue_features(h))) return rc;
    if (timed) (void)hipEventRecord(L->ev0, s);
    e = mlp_infer(L->mlp, s, L->d_feat, nv, L->d_corr);
    if (timed) (void)hipEventRecord(L->ev1, s);
    if (e != hipSuccess) return hip_err(h, e, "mlp launch");
    hipLaunchKernelGGL(k_apply_corr, dim3(nb(nv)), dim3(256), 0, s, h->d_pos, h->d_vel, L->d_corr, nv);
    if ((e = hipGetLastError()) != hipSuccess) return hip_err(h, e, "apply launch");
    const bool warm = L->start == XPBD_LEARNED_START_MULTIPLIERS;
    const bool consistent = L->start == XPBD_LEARNED_START_CONSISTENT;
    if (warm && (rc = enqueue_multiplier_start(h))) return rc;
    if (consistent && (rc = enqueue_consistent_start(h))) return rc;
    if ((rc = enqueue_iterations(h, iters, false, !(warm || consistent)))) return rc;
    e = launch_residual(s, tet_arrays(h), h->d_pos, h->d_lo, true, h->nt, h->d_part, h->red_blocks, nullptr);
    if (e == hipSuccess) e = launch_sum_partials(s, h->d_part, h->red_blocks, L->d_res);
    if (e != hipSuccess) return hip_err(h, e, "learned residual");
    if (records_residuals(h) && (rc = enqueue_step_residual(h))) return rc;
    if ((rc = enqueue_local_collision(h))) return rc;
    MotionSource from;
    from.pred = L->d_pred;
    from.cprev = L->d_cprev;
    return enqueue_finish(h, from);
}

// Launch the attempt from a captured graph (built on first use of its shape).
static int launch_learned_attempt(xpbd_handle* h, int32_t iters, bool det)
{
    Learned* L = h->learned;
    const uint64_t net = L->mlp->version;
    hipGraphExec_t exec = nullptr;
    for (size_t i = 0; i < L->graphs.size();) {
        Learned::Graph& g = L->graphs[i];
        if (g.gen != h->graph_gen) {  // the handle's captured steps went stale: so did this one
            (void)hipGraphExecDestroy(g.exec);
            L->graphs[i] = L->graphs.back();
            L->graphs.pop_back();
            continue;
        }
        if (g.net == net && g.det == (int)det && g.iters == iters && g.start == L->start) exec = g.exec;
        i++;
    }
    if (!exec) {
        hipError_t e = hipStreamBeginCapture(h->stream, hipStreamCaptureModeThreadLocal);
        if (e != hipSuccess) return hip_err(h, e, "hipStreamBeginCapture");
        int rc = enqueue_learned_attempt(h, iters, det, false);
        hipGraph_t g = nullptr;
        e = hipStreamEndCapture(h->stream, &g);
        if (rc) {
            if (g) (void)hipGraphDestroy(g);
            return rc;
        }
        if (e != hipSuccess) return hip_err(h, e, "hipStreamEndCapture");
        e = hipGraphInstantiate(&exec, g, nullptr, nullptr, 0);
        (void)hipGraphDestroy(g);
        if (e != hipSuccess) return hip_err(h, e, "hipGraphInstantiate");
        // graphs of other network versions are unlikely to be replayed again
        for (size_t i = 0; i < L->graphs.size();) {
            if (L->graphs[i].net != net) {
                (void)hipGraphExecDestroy(L->graphs[i].exec);
                L->graphs[i] = L->graphs.back();
                L->graphs.pop_back();
            } else {
                i++;
            }
        }
        L->graphs.push_back({ net, h->graph_gen, (int)det, iters, L->start, exec });
    }
    hipError_t e = hipGraphLaunch(exec, h->stream);
    return e == hipSuccess ? XPBD_OK : hip_err(h, e, "hipGraphLaunch");
}
}  // namespace xpbd

extern "C" int xpbd_step_learned(xpbd_handle* h, int32_t iters, double ref_residual, double fallback_ratio,
                                 int32_t* fell_back, double* residual)
{
    if (!h) return XPBD_E_INVALID_ARG;
    if (iters < 0 || !std::isfinite(ref_residual) || !std::isfinite(fallback_ratio))
        return set_err(h, XPBD_E_INVALID_ARG, "step_learned: iters >= 0 and finite thresholds required");
    if (!h->learned || !h->learned->mlp) return set_err(h, XPBD_E_STATE, "no network attached");
    Learned* L = h->learned;
    const int nv = h->nv;
    hipStream_t s = h->stream;
    const bool det = detect_this_step(h);
    // kernel timing mode launches eagerly and times the inference with events
    int rc = h->timing ? enqueue_learned_attempt(h, iters, det, true) : launch_learned_attempt(h, iters, det);
    if (rc) return rc;
    double r2 = 0;
    hipError_t e = hipMemcpyAsync(&r2, L->d_res, sizeof(double), hipMemcpyDeviceToHost, s);
    if (e == hipSuccess) e = hipStreamSynchronize(s);
    if (e != hipSuccess) return hip_err(h, e, "learned step");
    double r = std::sqrt(r2);
    if (h->timing) {
        float ms = 0.f;
        (void)hipEventElapsedTime(&ms, L->ev0, L->ev1);
        L->mlp_ms += ms;
        L->mlp_calls++;
    }
    const bool fb = ref_residual > 0 && fallback_ratio > 0 && !(r <= fallback_ratio * ref_residual);
    if (fb) {
        // redo the step from the snapshot as the plain solver does
        e = hipMemcpyAsync(h->d_pos, L->d_save, sizeof(float4) * 2 * (size_t)nv, hipMemcpyDeviceToDevice, s);
        if (e == hipSuccess)
            e = hipMemcpyAsync(h->d_lo, L->d_save + 2 * (size_t)nv, sizeof(float4) * nv, hipMemcpyDeviceToDevice, s);
        if (e == hipSuccess)
            e = hipMemcpyAsync(h->d_vel, L->d_save + 3 * (size_t)nv, sizeof(float4) * nv, hipMemcpyDeviceToDevice, s);
        if (e == hipSuccess)
            e = hipMemcpyAsync(h->d_step, L->d_step_save, sizeof(unsigned long long), hipMemcpyDeviceToDevice, s);
        if (e != hipSuccess) return hip_err(h, e, "learned restore");
        if ((rc = enqueue_predict(h)) || (rc = enqueue_copy_pred(h))) return rc;
        if ((rc = enqueue_iterations(h, h->params.iters, false))) return rc;
        if ((rc = device_residual(h, &r, nullptr))) return rc;
        if (records_residuals(h) && (rc = enqueue_step_residual(h))) return rc;
        if ((rc = enqueue_local_collision(h))) return rc;
        if ((rc = enqueue_store_cprev(h)) || (rc = enqueue_finish(h))) return rc;
        e = hipStreamSynchronize(s);
        if (e != hipSuccess) return hip_err(h, e, "learned fallback");
        L->fallbacks++;
    }
    h->host_step++;
    L->steps++;
    if (fell_back) *fell_back = fb ? 1 : 0;
    if (residual) *residual = r;
    return XPBD_OK;
}

extern "C" int xpbd_set_learned_start(xpbd_handle* h, int32_t mode)
{
    if (!h) return XPBD_E_INVALID_ARG;
    if (mode != XPBD_LEARNED_START_POSITIONS && mode != XPBD_LEARNED_START_MULTIPLIERS &&
        mode != XPBD_LEARNED_START_CONSISTENT)
        return set_err(h, XPBD_E_INVALID_ARG, "unknown learned start mode");
    int rc = ensure_learned(h);
    if (rc) return rc;
    if (mode == XPBD_LEARNED_START_CONSISTENT && (rc = ensure_vertex_slots(h))) return rc;
    h->learned->start = mode;
    return XPBD_OK;
}

extern "C" int xpbd_learned_stats(xpbd_handle* h, int64_t* steps, int64_t* fallbacks, double* mlp_ms,
                                  int64_t* mlp_calls)
{
    if (!h) return XPBD_E_INVALID_ARG;
    if (!h->learned) return set_err(h, XPBD_E_STATE, "no network attached");
    if (steps) *steps = h->learned->steps;
    if (fallbacks) *fallbacks = h->learned->fallbacks;
    if (mlp_ms) *mlp_ms = h->learned->mlp_ms;
    if (mlp_calls) *mlp_calls = h->learned->mlp_calls;
    return XPBD_OK;
}
