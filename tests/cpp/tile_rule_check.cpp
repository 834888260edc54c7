// Prints how many tile launches and how many colour launches a solve of ITERS
// iterations makes on the untuned default.
//   tile_rule_check NX NY NZ UNITS ITERS
#include <cstdio>
#include <cstdlib>
#include <vector>

#include "capi_internal.h"
#include "host_hip.h"
#include "mesh_tools.h"

using namespace xpbd;

static int tiles = 0, colours = 0;

namespace xpbd {
size_t gs_tile_smem(int slots, const GsTileShape& S)
{
    return S.lanes == 1 ? 16 * ((size_t)S.cap + slots) : 28 * (size_t)slots;
}
int gs_tile_cap(int slots) { return slots <= 1024 ? 1024 : slots <= 2048 ? 2048 : slots <= 4095 ? 4095 : 0; }
hipError_t launch_gs_tile(hipStream_t, const GsTileArgs&, const GsTileShape&, int, int, size_t, bool)
{
    return tiles++, hipSuccess;
}
hipError_t launch_gs_cluster_quad(hipStream_t, const TetArrays&, const int4*, const int*, const uint32_t*, float4*, int, int,
                                  bool, int, bool, int, float4*, const float4*)
{
    return colours++, hipSuccess;
}
}  // namespace xpbd

int main(int argc, char** argv)
{
    if (argc != 6) return 2;
    std::vector<double> x;
    std::vector<int32_t> t;
    const double o[3] = { 0, 0, 0 };
    grid_mesh(atoi(argv[1]), atoi(argv[2]), atoi(argv[3]), 0.01, 0.01, 0.01, o, x, t);
    const int nt = (int)(t.size() / 4);
    const std::vector<double> E(nt, 1000.0), nu(nt, 0.4);
    xpbd_mesh_desc d{};
    d.num_vertices = (int)(x.size() / 3);
    d.num_tets = nt;
    d.x0 = x.data();
    d.tets = t.data();
    d.E = d.rho = E.data();
    d.nu = nu.data();
    xpbd_params p{};
    p.dt = 1e-3;
    p.iters = 1;
    p.solver = XPBD_SOLVER_GS_COLORED;
    host_hip::units = atoi(argv[4]);
    xpbd_handle* h = nullptr;
    if (xpbd_create(&d, &p, &h) != XPBD_OK) return puts(xpbd_last_error(nullptr)), 1;
    if (enqueue_iterations(h, atoi(argv[5]), false)) return 1;
    printf("%d %d\n", tiles, colours);
    xpbd_destroy(h);
    return 0;
}
