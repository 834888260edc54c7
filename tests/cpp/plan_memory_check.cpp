// Host memory that runs out while a tile plan is built, at the n-th allocation and
// for all that follow until the call returns: the call has to return (an exception
// must not leave it, nor end a thread), with an error or a whole plan, and an error
// leaves the handle without a plan and gives the device memory back.
//   plan_memory_check SOLVER(gs|jacobi) NX NY NZ
#include <atomic>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <new>
#include <vector>

#include "capi_internal.h"
#include "host_hip.h"
#include "mesh_tools.h"

static std::atomic<int64_t> left{ INT64_MAX };   // allocations until there is no more
static std::atomic<int64_t> refused{ 0 };

void* operator new(size_t n)
{
    if (left.fetch_sub(1) <= 0) {
        refused++;
        throw std::bad_alloc();
    }
    if (void* p = std::malloc(n ? n : 1)) return p;
    throw std::bad_alloc();
}
void* operator new(size_t n, const std::nothrow_t&) noexcept
{
    if (left.fetch_sub(1) > 0) return std::malloc(n ? n : 1);
    refused++;
    return nullptr;
}
void operator delete(void* p) noexcept { std::free(p); }
void operator delete(void* p, size_t) noexcept { std::free(p); }

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
    const bool gs = std::strcmp(argv[1], "gs") == 0;
    std::vector<double> x;
    std::vector<int32_t> t;
    const double o[3] = { 0, 0, 0 };
    grid_mesh(atoi(argv[2]), atoi(argv[3]), atoi(argv[4]), 0.01, 0.01, 0.01, o, x, t);
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
    p.solver = gs ? XPBD_SOLVER_GS_COLORED : XPBD_SOLVER_JACOBI;
    p.deterministic = 1;
    p.variant = gs ? XPBD_VARIANT_CLUSTER_QUAD : XPBD_VARIANT_PATCH;   // no plan yet
    xpbd_handle* h = nullptr;
    if (xpbd_create(&d, &p, &h) != XPBD_OK) return puts(xpbd_last_error(nullptr)), 1;
    auto build = [&] { return gs ? ensure_gs_tiles(h) : ensure_jacobi_tiles(h); };
    auto planned = [&] { return gs ? !h->tiles.launches.empty() : h->jtiles.ready; };
    const size_t own = h->allocs.size();
    auto forget = [&] {
        for (; h->allocs.size() > own; h->allocs.pop_back()) (void)hipFree(h->allocs.back());
        h->tiles = GsTilePlan{};
        h->jtiles = JacobiTilePlan{};
    };
    const int64_t before = host_hip::device_bytes;
    int64_t errors = 0, bad = 0, n = 0;
    bool whole = false;
    for (; !whole && n < 1000000; n += 1 + n / 16) {
        std::fprintf(stderr, "%lld\n", (long long)n);   // where it ended, should it end
        refused = 0;
        left = n;
        const int rc = build();
        left = INT64_MAX;
        whole = refused == 0;
        errors += rc != XPBD_OK;
        bad += whole && !planned();
        bad += rc != XPBD_OK && (planned() || host_hip::device_bytes != before);
        forget();
        bad += host_hip::device_bytes != before;
    }
    printf("%lld refusals survived, up to allocation %lld, %lld wrong\n", (long long)errors, (long long)n, (long long)bad);
    xpbd_destroy(h);
    return bad != 0 || !whole || errors == 0;
}
