// Runs the vertex-tile Jacobi plan of a mesh on the CPU and compares it with the
// plain iteration.  Elements and faces give each of their vertices a hash of all
// their vertices' values, summed as integers.
// Each is added once, contacts by patch (LATE 0) or at the end.
//   jacobi_tiles_check NX NY NZ INSTANCES PARTS LATE
#include <algorithm>
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <vector>

#include "jacobi_tiles.h"
#include "mesh_tools.h"

using namespace xpbd;

static uint64_t mix(uint64_t h)
{
    h ^= h >> 31;
    h *= 0x9E3779B97F4A7C15ull;
    return h ^ (h >> 29);
}

static uint64_t part(uint64_t kind, int item, const uint64_t* v, int n, int k)
{
    uint64_t h = mix(kind + 1000003ull * item);
    for (int i = 0; i < n; i++) h = mix(h ^ v[i]);
    return mix(h + k);
}

int main(int argc, char** argv)
{
    if (argc != 7) return 2;
    const int patch = 16;
    const bool late = atoi(argv[6]) != 0;
    const int nx = atoi(argv[1]), ny = atoi(argv[2]), nz = atoi(argv[3]), ninst = atoi(argv[4]), parts = atoi(argv[5]);
    std::vector<double> x;
    std::vector<int32_t> t, faces, face_patch;
    std::vector<int64_t> v_off(1, 0);
    for (int i = 0; i < ninst; i++) {   // instances of different sizes, all at the origin
        std::vector<double> xi;
        std::vector<int32_t> ti;
        const double o[3] = { 0, 0, 0 };
        grid_mesh(nx + i, ny, nz + 2 * i, 0.01, 0.01, 0.01, o, xi, ti);
        const int32_t v0 = (int32_t)(x.size() / 3);
        for (int32_t v : ti) t.push_back(v + v0);
        x.insert(x.end(), xi.begin(), xi.end());
        v_off.push_back((int64_t)x.size() / 3);
        const int e0 = (int)(t.size() - ti.size()) / 4;
        for (size_t k = 0; k + 4 <= ti.size(); k += 12) {   // any triangles will do
            for (int32_t v : { ti[k] + v0, ti[k + 1] + v0, ti[k + 2] + v0, i }) faces.push_back(v);
            if (!late) face_patch.push_back((e0 + (int)k / 4) / patch);
        }
    }
    x.insert(x.end(), { 9.0, 9.0, 9.0 });   // a vertex of no element
    v_off.back()++;
    const int nv = (int)(x.size() / 3), nt = (int)(t.size() / 4), nf = (int)(faces.size() / 4);
    const JacobiMesh M{ nv, nt, nf, t.data(), faces.data(), patch, face_patch, v_off, x };
    JacobiTiles J;
    if (!build_jacobi_tiles(M, parts, 4, J)) return puts("no plan"), 1;
    std::vector<uint64_t> ref(nv), sum(nv);
    for (int v = 0; v < nv; v++) ref[v] = mix(v + 1);
    std::vector<uint64_t> d[2];
    for (auto& a : d) a.assign(J.vert.size(), 0);
    for (size_t s = 0; s < J.vert.size(); s++) d[0][s] = ref[J.vert[s]];
    std::vector<int> kept(nt, 0), kept_face(nf, 0);
    int64_t bad = 0;
    const int iters = 3;
    for (int it = 0; it < iters; it++) {
        std::fill(sum.begin(), sum.end(), 0);
        for (int e = 0; e < nt; e++) {
            uint64_t v[4];
            for (int k = 0; k < 4; k++) v[k] = ref[t[4 * (size_t)e + k]];
            for (int k = 0; k < 4; k++) sum[t[4 * (size_t)e + k]] += part(1, e, v, 4, k);
        }
        for (int f = 0; f < nf; f++) {
            uint64_t v[3];
            for (int k = 0; k < 3; k++) v[k] = ref[faces[4 * (size_t)f + k]];
            for (int k = 0; k < 3; k++) sum[faces[4 * (size_t)f + k]] += part(2, f, v, 3, k);
        }
        for (int v = 0; v < nv; v++) ref[v] = mix(ref[v] + sum[v]);
        for (int g = 0; g < J.ntiles; g++) {
            const int32_t* h = &J.head[(size_t)JacobiTiles::kHead * g];
            const uint64_t* l = &d[it & 1][h[JacobiTiles::V0]];
            std::vector<uint64_t> red(J.slots, 0), own(h[JacobiTiles::OWN]);
            std::vector<char> used(J.slots, 0);
            auto write = [&](int s, uint64_t x) {
                if (s == 0xffff) return;
                bad += s >= J.slots || used[s];
                used[s] = 1;
                red[s] = x;
            };
            for (int i = h[JacobiTiles::T0]; i < h[JacobiTiles::T0] + h[JacobiTiles::NT]; i++) {
                const uint16_t* a = &J.local[8 * (size_t)i];
                uint64_t v[4];
                for (int k = 0; k < 4; k++) {
                    bad += a[k] >= h[JacobiTiles::NV];
                    v[k] = l[a[k]];
                }
                for (int k = 0; k < 4; k++) write(a[4 + k], part(1, J.home[i] >> 1, v, 4, k));
                if (it == 0) kept[J.home[i] >> 1] += J.home[i] & 1;
            }
            for (int i = h[JacobiTiles::F0]; i < h[JacobiTiles::F0] + h[JacobiTiles::NF]; i++) {
                const uint32_t* a = (const uint32_t*)&J.face[4 * (size_t)i];
                const uint64_t v[3] = { l[a[1] & 0xffff], l[a[1] >> 16], l[a[2] & 0xffff] };
                const int s[3] = { (int)(a[2] >> 16), (int)(a[3] & 0xffff), (int)(a[3] >> 16) };
                for (int k = 0; k < 3; k++) write(s[k], part(2, (int)a[0] >> 1, v, 3, k));
                if (it == 0) kept_face[a[0] >> 1] += a[0] & 1;
            }
            for (int o = 0; o < h[JacobiTiles::OWN]; o++) {
                const uint32_t* q = &J.sums[JacobiTiles::kSums * (size_t)(h[JacobiTiles::V0] + o)];
                const uint64_t end = q[0] | (uint64_t)q[1] << 32, con = q[2] | (uint64_t)q[3] << 32;
                const int32_t* gr = &J.group[2 * (size_t)(h[JacobiTiles::G0] + o / 64)];
                uint64_t s = 0, part = 0;
                uint32_t f = 0;
                auto contacts = [&] {
                    for (bool more = true; more; f++) {
                        s += red[gr[1] + 64 * f + o % 64];
                        more = !(q[5] >> f & 1);
                    }
                };
                for (uint32_t e = 0; e < (q[4] & 0xffff); e++) {
                    part += red[gr[0] + 64 * e + o % 64];
                    if (con >> e & 1) contacts();
                    if (end >> e & 1) {
                        s += part;
                        part = 0;
                    }
                }
                if (late && q[4] >> 16) contacts();
                bad += part != 0 || f != q[4] >> 16;
                own[o] = mix(l[o] + s);
            }
            for (int k = h[JacobiTiles::O0]; k < h[JacobiTiles::O0] + h[JacobiTiles::NO]; k++)
                d[1 - (it & 1)][J.out[2 * (size_t)k + 1]] = own[J.out[2 * (size_t)k]];
        }
    }
    for (size_t s = 0; s < J.vert.size(); s++) bad += d[iters & 1][s] != ref[J.vert[s]];
    for (int v = 0; v < nv; v++) bad += d[iters & 1][J.owner[v]] != ref[v];
    for (int k : kept) bad += k != 1;
    for (int k : kept_face) bad += k != 1;
    printf("%d tiles, %.2f copies of an element, closed %d, wrong %lld\n", J.ntiles, (double)J.home.size() / nt,
           (int)J.closed, (long long)bad);
    return bad != 0;
}
