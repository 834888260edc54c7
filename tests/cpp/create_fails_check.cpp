// Device memory that runs out while a handle is created, at the n-th allocation, with
// the plan's host work under way on its thread: the creation fails, or goes on without
// what it can do without, and nothing is left behind.
//   create_fails_check SOLVER(gs|jacobi) NX NY NZ
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <vector>

#include "capi_internal.h"
#include "host_hip.h"
#include "mesh_tools.h"

using namespace xpbd;

namespace xpbd {
size_t gs_tile_smem(int slots, const GsTileShape& S)
{
    return S.lanes == 1 ? 16 * ((size_t)S.cap + slots) : 28 * (size_t)slots;
}
int gs_tile_cap(int slots) { return slots <= 1024 ? 1024 : slots <= 2048 ? 2048 : slots <= 4095 ? 4095 : 0; }
size_t jacobi_tile_smem(int verts, int slots) { return 32 * (size_t)verts + 12 * (size_t)slots + 2048; }
}  // namespace xpbd

int main(int argc, char** argv)
{
    if (argc != 5) return 2;
    std::vector<double> x;
    std::vector<int32_t> t, f;
    const double o[3] = { 0, 0, 0 };
    grid_mesh(atoi(argv[2]), atoi(argv[3]), atoi(argv[4]), 0.01, 0.01, 0.01, o, x, t);
    const int nt = (int)(t.size() / 4);
    surface_faces((int)(x.size() / 3), nt, t.data(), f);
    const std::vector<double> E(nt, 1000.0), nu(nt, 0.4);
    xpbd_mesh_desc d{};
    d.num_vertices = (int)(x.size() / 3);
    d.num_tets = nt;
    d.x0 = x.data();
    d.tets = t.data();
    d.E = d.rho = E.data();
    d.nu = nu.data();
    d.num_faces = (int)(f.size() / 3);
    d.faces = f.data();
    xpbd_params p{};
    p.dt = 1e-3;
    p.iters = 1;
    p.solver = std::strcmp(argv[1], "gs") == 0 ? XPBD_SOLVER_GS_COLORED : XPBD_SOLVER_JACOBI;
    p.deterministic = 1;
    int64_t bad = 0, refused = 0, plain = 0;
    for (int64_t n = 0;; n++) {
        host_hip::mallocs = 0;
        host_hip::mallocs_left = n;
        xpbd_handle* h = nullptr;
        const int rc = xpbd_create(&d, &p, &h);
        const bool whole = host_hip::mallocs_left >= 0;
        bad += rc == XPBD_OK ? !h : h != nullptr || rc != XPBD_E_NOMEM;
        refused += rc != XPBD_OK;
        if (h) {
            const bool tiles = !h->tiles.launches.empty() || h->jtiles.ready;
            bad += whole && !tiles;
            plain += !tiles;
            xpbd_destroy(h);
        }
        bad += host_hip::device_bytes != 0;
        if (whole) break;
    }
    printf("%lld refused, %lld without tiles, %lld wrong\n", (long long)refused, (long long)plain, (long long)bad);
    return bad != 0 || refused == 0 || plain == 0;
}
