// The quad shape that colour launches get on a handle whose autotune, or whose cache
// file PATH, chose the fused-colour launches, with an attachment.
//   tuned_shape_check PATH
// Prints the choice and that shape before, then after the autotune.
#include <cstdio>
#include <vector>

#include "capi_internal.h"
#include "host_hip.h"
#include "mesh_tools.h"

using namespace xpbd;

static int shape = 0;

namespace xpbd {
size_t gs_tile_smem(int slots, const GsTileShape& S)
{
    return S.lanes == 1 ? 16 * ((size_t)S.cap + slots) : 28 * (size_t)slots;
}
int gs_tile_cap(int slots) { return slots <= 1024 ? 1024 : slots <= 2048 ? 2048 : slots <= 4095 ? 4095 : 0; }
hipError_t launch_gs_cluster_quad(hipStream_t, const TetArrays&, const int4*, const int*, const uint32_t*, float4*, int, int,
                                  bool, int block, bool, int, float4*, const float4*)
{
    return shape = block, hipSuccess;
}
}  // namespace xpbd

int main(int argc, char** argv)
{
    if (argc != 2) return 2;
    std::vector<double> x;
    std::vector<int32_t> t;
    const double o[3] = { 0, 0, 0 };
    grid_mesh(9, 9, 9, 0.01, 0.01, 0.01, o, x, t);
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
    p.iters = 2;
    p.solver = XPBD_SOLVER_GS_COLORED;
    xpbd_handle* h = nullptr;
    if (xpbd_create(&d, &p, &h) != XPBD_OK) return puts(xpbd_last_error(nullptr)), 1;
    const int32_t v = 0;
    for (int tuned = 0; tuned < 2; tuned++) {
        if (tuned && xpbd_autotune(h, argv[1]) != XPBD_OK) return puts(xpbd_last_error(h)), 1;
        int32_t variant = 0, block = 0;
        xpbd_get_variant(h, &variant, &block, nullptr);
        if (xpbd_set_attachments(h, 1, &v, x.data()) || enqueue_iterations(h, 2, false)) return 1;
        printf("%d %d %d\n", variant, block, shape);
        if (xpbd_set_attachments(h, 0, nullptr, nullptr)) return 1;
    }
    xpbd_destroy(h);
    return 0;
}
