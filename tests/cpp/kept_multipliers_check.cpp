// A warm-started solve's multipliers through the tile launches that the host code
// makes for it, run on the CPU with each projection replaced by adding one.  A
// launch's tiles run one after the other, forwards or backwards: whatever the order,
// every copy of an element has to start from the multipliers that the solve was
// given, and every element has to end with theirs plus the iterations.
//   kept_multipliers_check SOLVER(gs|jacobi) NX NY NZ INSTANCES UNITS
#include <algorithm>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <vector>

#include "capi_internal.h"
#include "host_hip.h"
#include "jacobi_tiles.h"
#include "mesh_tools.h"

using namespace xpbd;

namespace {
std::vector<GsTileFill> fills;       // of each group, in order
const int32_t* cstart = nullptr;
bool backwards = false;
int64_t wrong = 0, launches = 0, tiles = 0;
std::vector<float> given;            // per element, what the solve starts from

int tile_at(int i, int n) { return backwards ? n - 1 - i : i; }

float started(bool first, bool zero, float kept, float own, int e, int it)
{
    const float x = first ? (zero ? 0.f : kept) : own;
    wrong += x != given[e] + (float)it;
    return x;
}
}  // namespace

namespace xpbd {

size_t gs_tile_smem(int slots, const GsTileShape& S)
{
    return S.lanes == 1 ? 16 * ((size_t)S.cap + slots) : 28 * (size_t)slots;
}
int gs_tile_cap(int slots) { return slots <= 1024 ? 1024 : slots <= 2048 ? 2048 : slots <= 4095 ? 4095 : 0; }
hipError_t launch_gs_tile_fill(hipStream_t, const GsTileFill& A, const GsTileShape&)
{
    fills.push_back(A);
    cstart = A.cstart;
    return hipSuccess;
}
// A copy's own multipliers: here at 8 per place of clu, which the arrays of both kernels have room for.
hipError_t launch_gs_tile(hipStream_t, const GsTileArgs& A, const GsTileShape& S, int ntiles, int, size_t, bool import)
{
    static std::vector<std::vector<float>> lam(64);
    static int iteration = 0;
    size_t g = 0;
    while (fills[g].lam != A.lam) g++;
    const GsTileFill& F = fills[g];
    const int per = S.lanes == 1 ? 64 : 16, blocks = F.nblocks / ntiles;
    lam[g].resize(8 * (size_t)per * F.nblocks);
    if (A.lam_zero || import) iteration = 0;
    launches++;
    tiles = ntiles;
    for (int i = 0; i < ntiles; i++) {
        const int t = tile_at(i, ntiles);
        for (int c = t * blocks * per; c < (t + 1) * blocks * per; c++) {
            if (F.clu[c] < 0) continue;
            const int e0 = cstart[F.clu[c]], n = cstart[F.clu[c] + 1] - e0;
            for (int k = 0; k < n; k++) {
                float& own = lam[g][8 * (size_t)c + k];
                float x = started(A.lam_zero || import, A.lam_zero, A.kept ? A.kept[e0 + k].x : 0.f, own, e0 + k, iteration);
                for (int it = 0; it < A.niter; it++) x += 1.f;
                own = x;
                if (A.lam_out && F.own[c]) A.dlam[e0 + k].x = x;
            }
        }
    }
    if (g + 1 == fills.size()) iteration += A.niter;
    return hipSuccess;
}

size_t jacobi_tile_smem(int verts, int slots) { return 32 * (size_t)verts + 12 * (size_t)slots + 2048; }
hipError_t launch_jacobi_tile(hipStream_t, const JacobiTileArgs& A, int, bool)
{
    static int iteration = 0;
    if (A.lam_zero || A.import) iteration = 0;
    launches++;
    tiles = A.ntiles;
    for (int i = 0; i < A.ntiles; i++) {
        const int* h = A.head + JacobiTiles::kHead * tile_at(i, A.ntiles);
        for (int e = h[JacobiTiles::T0]; e < h[JacobiTiles::T0] + h[JacobiTiles::NT]; e++) {
            const int at = A.home[e] >> 1;
            float x = started(A.lam_zero || A.import, A.lam_zero, A.kept ? A.kept[at].x : 0.f, A.lam[e].x, at, iteration);
            for (int it = 0; it < A.niter; it++) x += 1.f;
            A.lam[e].x = x;
            if (A.lam_out && (A.home[e] & 1)) A.dlam[at].x = x;
        }
    }
    iteration += A.niter;
    return hipSuccess;
}

}  // namespace xpbd

int main(int argc, char** argv)
{
    if (argc != 7) return 2;
    const int ninst = atoi(argv[5]);
    host_hip::units = atoi(argv[6]);
    std::vector<std::vector<double>> x(ninst), m(ninst);
    std::vector<std::vector<int32_t>> t(ninst);
    std::vector<xpbd_mesh_desc> d(ninst);
    for (int i = 0; i < ninst; i++) {
        const double o[3] = { 0, 0, 0 };
        grid_mesh(atoi(argv[2]) + i, atoi(argv[3]), atoi(argv[4]) + 2 * i, 0.01, 0.01, 0.01, o, x[i], t[i]);
        const int nt = (int)(t[i].size() / 4);
        m[i].assign(3 * (size_t)nt, 1000.0);
        std::fill(m[i].begin() + nt, m[i].begin() + 2 * nt, 0.4);
        d[i] = {};
        d[i].num_vertices = (int)(x[i].size() / 3);
        d[i].num_tets = nt;
        d[i].x0 = x[i].data();
        d[i].tets = t[i].data();
        d[i].E = m[i].data();
        d[i].nu = m[i].data() + nt;
        d[i].rho = m[i].data() + 2 * nt;
    }
    xpbd_params p{};
    p.dt = 1e-3;
    p.iters = 3;
    p.solver = std::strcmp(argv[1], "gs") == 0 ? XPBD_SOLVER_GS_COLORED : XPBD_SOLVER_JACOBI;
    p.deterministic = 1;
    xpbd_handle* h = nullptr;
    if (xpbd_batch_create(ninst, d.data(), &p, &h) != XPBD_OK) return puts(xpbd_last_error(nullptr)), 1;
    given.resize(h->nt);
    int64_t bad = 0;
    for (int iters : { 1, 2, 3, 1 })
        for (int back = 0; back < 2; back++)
            for (int reset = 0; reset < 2; reset++) {
                backwards = back != 0;
                for (int e = 0; e < h->nt; e++) {
                    h->d_lam[e] = make_float2((float)(1 + e % 1000), 0.f);
                    given[e] = reset ? 0.f : h->d_lam[e].x;
                }
                wrong = launches = 0;
                if (enqueue_iterations(h, iters, false, reset != 0)) return puts("enqueue"), 1;
                int64_t ends = 0;
                for (int e = 0; e < h->nt; e++) ends += h->d_lam[e].x != given[e] + (float)iters;
                if (wrong || ends)
                    printf("%d iterations%s%s: %lld wrong starts, %lld wrong ends\n", iters, back ? ", backwards" : "",
                           reset ? "" : ", kept", (long long)wrong, (long long)ends);
                bad += wrong + ends + (launches == 0);
            }
    printf("%lld tiles, %lld launches\n", (long long)tiles, (long long)launches);
    xpbd_destroy(h);
    return bad != 0 || host_hip::device_bytes != 0;
}
