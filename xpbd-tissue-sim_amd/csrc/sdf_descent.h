// Signed distances of the colliders and the closest-point search on a face, in
// FP64 without FMA contraction (see solver_kernels.hip), for the device and,
// compiled with -ffp-contract=off, for the host.
//
// SphereSDF.cpp:16-26, BoxSDF.cpp:19-84, GeometryUtils.cpp:6-24,92-102,
// CollisionScene.cpp:253-283 (Frank-Wolfe).
#pragma once
#include <cmath>

#ifdef __HIPCC__
#define XPBD_HD __host__ __device__ __forceinline__
#else
#define XPBD_HD inline
#endif
#ifdef __clang__
#pragma clang fp contract(off)
#endif

namespace xpbd {

struct Pose {
    int kind;   // 1 sphere, else box
    double p[3], q[4], prm[3];
};

XPBD_HD void qrot(const double* v, const double* q, double* o)
{
    const double uv = q[0] * v[0] + q[1] * v[1] + q[2] * v[2];
    const double cx = q[1] * v[2] - q[2] * v[1];
    const double cy = q[2] * v[0] - q[0] * v[2];
    const double cz = q[0] * v[1] - q[1] * v[0];
    const double s = 2 * q[3] * q[3] - 1;
    o[0] = 2 * uv * q[0] + s * v[0] + 2 * q[3] * cx;
    o[1] = 2 * uv * q[1] + s * v[1] + 2 * q[3] * cy;
    o[2] = 2 * uv * q[2] + s * v[2] + 2 * q[3] * cz;
}

// a collider and, for a box, the inverse rotation
struct PosedSdf : Pose {
    double n2, qi[4];

    XPBD_HD explicit PosedSdf(const Pose& P) : Pose(P), n2(1.0), qi{}
    {
        if (kind == 1) return;
        n2 = q[0] * q[0] + q[1] * q[1] + q[2] * q[2] + q[3] * q[3];
        qi[0] = -q[0] / n2;
        qi[1] = -q[1] / n2;
        qi[2] = -q[2] / n2;
        qi[3] = q[3] / n2;
    }
};

XPBD_HD void to_body(const PosedSdf& P, const double* x, double* xb)
{
    const double rel[3] = { x[0] - P.p[0], x[1] - P.p[1], x[2] - P.p[2] };
    qrot(rel, P.qi, xb);
}

XPBD_HD double sdf_eval(const PosedSdf& P, const double* x)
{
    if (P.kind == 1) {
        const double d0 = x[0] - P.p[0], d1 = x[1] - P.p[1], d2 = x[2] - P.p[2];
        return sqrt(d0 * d0 + d1 * d1 + d2 * d2) - P.prm[0];
    }
    double xb[3];
    to_body(P, x, xb);
    double q[3], qc[3];
#pragma unroll
    for (int k = 0; k < 3; k++) {
        q[k] = fabs(xb[k]) - 0.5 * P.prm[k];
        qc[k] = q[k] > 0.0 ? q[k] : 0.0;
    }
    const double mq = fmax(q[0], fmax(q[1], q[2]));
    return sqrt(qc[0] * qc[0] + qc[1] * qc[1] + qc[2] * qc[2]) + (mq < 0.0 ? mq : 0.0);
}

XPBD_HD void sdf_grad(const PosedSdf& P, const double* x, double* g)
{
    if (P.kind == 1) {
        const double d[3] = { x[0] - P.p[0], x[1] - P.p[1], x[2] - P.p[2] };
        const double n = sqrt(d[0] * d[0] + d[1] * d[1] + d[2] * d[2]);
#pragma unroll
        for (int k = 0; k < 3; k++) g[k] = n > 0 ? d[k] / n : d[k];
        return;
    }
    double xb[3];
    to_body(P, x, xb);
    double q[3], qc[3], sg[3];
#pragma unroll
    for (int k = 0; k < 3; k++) {
        q[k] = fabs(xb[k]) - P.prm[k] / 2.0;
        qc[k] = q[k] > 0.0 ? q[k] : 0.0;
        sg[k] = xb[k] > 0 ? 1.0 : -1.0;
    }
    const double mq = fmax(q[0], fmax(q[1], q[2]));
    const double md = mq < 0.0 ? mq : 0.0;
    double go[3] = { sg[0] * qc[0], sg[1] * qc[1], sg[2] * qc[2] };
    const double n = sqrt(go[0] * go[0] + go[1] * go[1] + go[2] * go[2]);
    if (n > 0) {
#pragma unroll
        for (int k = 0; k < 3; k++) go[k] /= n;
    }
    double gb[3];
#pragma unroll
    for (int k = 0; k < 3; k++) gb[k] = go[k] + sg[k] * (q[k] == md ? 1.0 : 0.0);
    qrot(gb, P.q, g);
}

// ---------------------------------------------------------------------------
// Frank-Wolfe, 32 steps of size 2/(i+3): step i moves towards the vertex whose
// dot product with the gradient at x is least.  Only which vertex that is
// counts, so a step first forms the dot products of the face's edges with a
// positive multiple of the gradient, without the square root, the divisions and
// the rotation back, and calls sdf_grad only if their signs are not certain.
//
// Bounds, with eps = 2^-53, X the largest 1-norm of a vertex, R that of a vertex
// from the collider's centre, H of the half extents, v the multiple:
//   sphere  v = x - centre is the gradient's own, and the gradient is v / |v| to
//           4 eps a component.  A difference of two of its dot products is then
//           within 14 eps X of the exact one; the edges' rounding and their dot
//           products are within 10 eps X |v|.
//   box     y = x in the box's frame by the rotation's matrix: within 300 eps R
//           of to_body(x) (|q|^2 within 1e-3 of 1), and |y| - h within
//           tau = 2^-42 (R + X + H) of the exact code's.  Where no |y| - h is
//           within tau of a change of its case (outside: zero; inside: the
//           largest, and of the zero that its sign depends on), both take the
//           same case, and v, in the box's frame, is within tau a component.  The
//           edges, rotated into that frame, and their dot products are within
//           440 eps X |v| + 6 tau X.
// The margin X (2^-42 |v| + 8 tau), 2048 eps, is above the sums.  Ranges of 1e-140
// to 1e140, for a sphere's v by its margin's last term, keep squares and products
// clear of underflow and overflow; what is not a number fails its comparison.
// ---------------------------------------------------------------------------
template <bool BOX>
struct FaceDescent {
    double e1[3], e2[3];   // edges from the first vertex, for a box in its frame
    double N[3][3];        // box: its inverse rotation
    double h[3], tau;      // box: half extents
    double ms, m0;         // margin: ms |v| + m0
    int ok;                // ranges as above

    XPBD_HD FaceDescent(const PosedSdf& P, const double* p1, const double* p2, const double* p3)
    {
        const double* pv[3] = { p1, p2, p3 };
        double X = 0.0, R = 0.0, u[3][3];
#pragma unroll
        for (int j = 0; j < 3; j++) {
            double a = 0.0, r = 0.0;
#pragma unroll
            for (int k = 0; k < 3; k++) {
                u[j][k] = pv[j][k];
                a += fabs(pv[j][k]);
                r += fabs(pv[j][k] - P.p[k]);
            }
            X = fmax(X, a);
            R = fmax(R, r);
        }
        ok = (int)(X > 1e-140) & (int)(X < 1e140) & (int)(R < 1e140);
        ms = X * 0x1p-42;
        m0 = X * 1e-130;
        if constexpr (BOX) {
            const double qt[4] = { -P.q[0], -P.q[1], -P.q[2], P.q[3] };   // the transposed rotation
            double H = 0.0;
#pragma unroll
            for (int k = 0; k < 3; k++) {
                const double e[3] = { k == 0 ? 1.0 : 0.0, k == 1 ? 1.0 : 0.0, k == 2 ? 1.0 : 0.0 };
                double c[3];
                qrot(pv[k], qt, u[k]);
                qrot(e, P.qi, c);
#pragma unroll
                for (int i = 0; i < 3; i++) N[i][k] = c[i];
                h[k] = P.prm[k] / 2.0;
                H += fabs(h[k]);
            }
            tau = 0x1p-42 * (R + X + H);
            m0 = 8.0 * X * tau;
            ok &= (int)(H < 1e140) & (int)(fabs(P.n2 - 1.0) < 1e-3);
        }
#pragma unroll
        for (int k = 0; k < 3; k++) {
            e1[k] = u[1][k] - u[0][k];
            e2[k] = u[2][k] - u[0][k];
        }
    }

    // the vertex of the least dot product at x: 0, 1, 2, or -1 if too close to tell.  Conditions are
    // joined without short cuts: a branch costs a wave more than the comparison.
    XPBD_HD int vertex(const PosedSdf& P, const double* x) const
    {
        double v[3];
        int sure = ok;
#pragma unroll
        for (int k = 0; k < 3; k++) v[k] = x[k] - P.p[k];
        if constexpr (BOX) {
            double y[3], q[3];
#pragma unroll
            for (int k = 0; k < 3; k++) {
                y[k] = fma(N[k][2], v[2], fma(N[k][1], v[1], N[k][0] * v[0]));
                q[k] = fabs(y[k]) - h[k];
            }
            const double mq = fmax(q[0], fmax(q[1], q[2]));
            const int in = mq < 0.0;
            const double above = in ? mq - 2.0 * tau : 0.0;   // inside: only one may be
            int a[3];
            sure &= fabs(mq) > tau;
#pragma unroll
            for (int k = 0; k < 3; k++) {
                a[k] = q[k] > above;
                sure &= (int)((in ? fabs(y[k]) : fabs(q[k])) > tau) | (in & (a[k] ^ 1));
                v[k] = a[k] ? copysign(in ? 1.0 : q[k], y[k]) : 0.0;
            }
            sure &= (in ^ 1) | ((a[0] ^ a[1] ^ a[2]) & ((a[0] & a[1]) ^ 1));
        }
        const double m = fma(ms, fabs(v[0]) + fabs(v[1]) + fabs(v[2]), m0);
        const double a = fma(e1[2], v[2], fma(e1[1], v[1], e1[0] * v[0]));
        const double b = fma(e2[2], v[2], fma(e2[1], v[1], e2[0] * v[0]));
        const double c = b - a;
        const int c0 = (int)(a > m) & (int)(b > m), c1 = (int)(-a > m) & (int)(c > m),
                  c2 = (int)(-b > m) & (int)(-c > m);
        return ((sure & (c0 | c1 | c2)) - 1) | c1 | c2 << 1;
    }
};

struct FwSteps {
    double a[33];
    constexpr FwSteps() : a()
    {
        for (int i = 0; i < 33; i++) a[i] = 2.0 / (i + 3);
    }
};

// A wave pays for both choices where a lane is not sure.  Faces parallel to a box's tie at
// every step: after that many such steps the wave goes on with the plain choice alone
// (259,200 faces inside aligned boxes: 88 -> 71 us, the plain choice in all steps 67).
// Over a sphere ties pass with a step or two, and giving up costs more (15 -> 17 us).
constexpr int kQuickTries = 2;

// x: the vertex to start at, then the point found.  Returns the steps that took sdf_grad.
template <bool BOX, bool QUICK>
XPBD_HD int face_descent(const PosedSdf& P, const double* p1, const double* p2, const double* p3, double* x)
{
    constexpr FwSteps steps{};
    const FaceDescent<BOX> D(P, p1, p2, p3);
    int plain = 0, tries = kQuickTries;
    double al = steps.a[0];
#pragma unroll 1
    for (int it = 0; it < 32; it++) {
        const double next = steps.a[it + 1];   // on its way while this step is worked out
        int j = QUICK && tries > 0 ? D.vertex(P, x) : -1;
#ifdef __HIP_DEVICE_COMPILE__
        if (BOX && QUICK && tries > 0 && __any(j < 0)) tries--;   // of the wave: the same in every lane
#endif
        if (j < 0) {
            double g[3];
            sdf_grad(P, x, g);
            const double s1 = p1[0] * g[0] + p1[1] * g[1] + p1[2] * g[2];
            const double s2 = p2[0] * g[0] + p2[1] * g[1] + p2[2] * g[2];
            const double s3 = p3[0] * g[0] + p3[1] * g[1] + p3[2] * g[2];
            j = (s1 < s2 && s1 < s3) ? 0 : ((s2 < s1 && s2 < s3) ? 1 : 2);
            plain++;
        }
#pragma unroll
        for (int k = 0; k < 3; k++) x[k] = x[k] + al * ((j == 0 ? p1[k] : j == 1 ? p2[k] : p3[k]) - x[k]);
        al = next;
    }
    return plain;
}

}  // namespace xpbd
