// The closest-point search with its quick vertex choice against the plain one,
// bit for bit, over colliders and faces of many kinds.
#include <cmath>
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <limits>
#include <random>

#include "sdf_descent.h"

using namespace xpbd;

int main(int argc, char** argv)
{
    if (argc != 4) return 2;
    const int kind = atoi(argv[1]), mode = atoi(argv[2]), n = atoi(argv[3]);
    std::mt19937_64 rng(1000 * kind + mode);
    std::uniform_real_distribution<double> U(-1.0, 1.0);
    std::normal_distribution<double> N;
    long long plain = 0, bad = 0;
    for (int i = 0; i < n; i++) {
        Pose P{};
        P.kind = kind;
        double p[3][3];
        // a face with edges of some 0.01 near the collider's surface
        double far = mode == 1 ? 100.0 : mode == 2 ? 1e-6 : 1.0, edge = mode == 2 ? 1e-8 : 0.01;
        for (int k = 0; k < 3; k++) P.p[k] = far * U(rng);
        for (int k = 0; k < 4; k++) P.q[k] = N(rng);
        const double s = std::sqrt(P.q[0] * P.q[0] + P.q[1] * P.q[1] + P.q[2] * P.q[2] + P.q[3] * P.q[3]);
        for (int k = 0; k < 4; k++) P.q[k] /= s;
        for (int k = 0; k < 3; k++) P.prm[k] = mode == 2 ? 1e-8 * (1.5 + U(rng)) : 0.02 * (1.5 + U(rng));
        for (int j = 0; j < 3; j++)
            for (int k = 0; k < 3; k++) p[j][k] = P.p[k] + edge * 2 * U(rng);
        if (mode == 3 || mode == 4) {   // everything on a grid: symmetric faces, edges and medial planes; unrotated boxes
            for (int k = 0; k < 4; k++) P.q[k] = k == (mode == 3 ? 3 : (int)(rng() % 4));
            for (int k = 0; k < 3; k++) {
                P.p[k] = 0.01 * (double)(int)(rng() % 5);
                P.prm[k] = 0.01 * (double)(int)(rng() % 4);
                for (int j = 0; j < 3; j++) p[j][k] = 0.01 * (double)(int)(rng() % 5) + (mode == 4 ? 1e-16 * U(rng) : 0.0);
            }
        }
        if (mode == 5)   // not a unit quaternion, sizes of zero and less
            for (int k = 0; k < 4; k++) {
                P.q[k] *= 1.0 + 0.002 * U(rng) * (double)(rng() % 3);
                if (k < 3 && rng() % 4 == 0) P.prm[k] = rng() % 2 ? 0.0 : -0.01;
            }
        if (mode == 6) {   // scales from underflow to overflow, and what is no number
            const double scale = std::pow(10.0, 320.0 * U(rng));
            for (int k = 0; k < 3; k++) {
                P.p[k] *= scale;
                P.prm[k] *= rng() % 2 ? scale : 1.0;
                for (int j = 0; j < 3; j++) p[j][k] *= rng() % 8 ? scale : 1.0;
            }
            if (rng() % 4 == 0) p[rng() % 3][rng() % 3] = rng() % 2 ? std::numeric_limits<double>::infinity() : std::nan("");
            if (rng() % 8 == 0) P.q[rng() % 4] = rng() % 2 ? 1e200 : std::nan("");
        }
        if (mode == 7)   // a vertex, an edge's middle or the face's in the collider's centre
            for (int k = 0; k < 3; k++) P.p[k] = i % 3 == 0 ? p[0][k] : i % 3 == 1 ? (p[0][k] + p[1][k]) / 2 : (p[0][k] + p[1][k] + p[2][k]) / 3;
        const int st = (int)(rng() % 3);
        double a[3], b[3];
        for (int k = 0; k < 3; k++) a[k] = b[k] = p[st][k];
        const PosedSdf S(P);
        if (kind == 1) {
            plain += face_descent<false, true>(S, p[0], p[1], p[2], a);
            face_descent<false, false>(S, p[0], p[1], p[2], b);
        } else {
            plain += face_descent<true, true>(S, p[0], p[1], p[2], a);
            face_descent<true, false>(S, p[0], p[1], p[2], b);
        }
        for (int k = 0; k < 3; k++)
            if (std::memcmp(&a[k], &b[k], 8) != 0 && !(std::isnan(a[k]) && std::isnan(b[k]))) bad++;
    }
    printf("%lld wrong, %.4f of the steps by the plain choice\n", bad, (double)plain / (32.0 * n));
    return bad != 0;
}
