// Device memory of a batch of COUNT cubes of SMALL cells per axis and one of LARGE, with
// or without faces, of which PLAN is what the untuned default holds beyond a handle
// without tiles, and CONTACTS what faces add.  Prints both in bytes, whether all colours
// share a launch, and the vertices; then those of a batch of UNITS cubes of LARGE.
//   uneven_batch_check SMALL COUNT LARGE UNITS
#include <cstdio>
#include <cstdlib>
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
}  // namespace xpbd

struct Cube {
    std::vector<double> x, E, nu;
    std::vector<int32_t> t, f;
    explicit Cube(int n)
    {
        const double o[3] = { 0, 0, 0 };
        grid_mesh(n, n, n, 0.01, 0.01, 0.01, o, x, t);
        E.assign(t.size() / 4, 1000.0);
        nu.assign(t.size() / 4, 0.4);
        surface_faces((int)(x.size() / 3), (int)(t.size() / 4), t.data(), f);
    }
    xpbd_mesh_desc desc(bool faces) const
    {
        xpbd_mesh_desc d{};
        d.num_vertices = (int)(x.size() / 3);
        d.num_tets = (int)(t.size() / 4);
        d.x0 = x.data();
        d.tets = t.data();
        d.E = d.rho = E.data();
        d.nu = nu.data();
        if (faces) d.faces = f.data();
        d.num_faces = faces ? (int)(f.size() / 3) : 0;
        return d;
    }
};

static int64_t held(const std::vector<xpbd_mesh_desc>& d, int variant, bool* planned)
{
    xpbd_params p{};
    p.dt = 1e-3;
    p.iters = 3;
    p.solver = XPBD_SOLVER_GS_COLORED;
    p.variant = variant;
    xpbd_handle* h = nullptr;
    if (xpbd_batch_create((int)d.size(), d.data(), &p, &h) != XPBD_OK) {
        puts(xpbd_last_error(nullptr));
        exit(1);
    }
    const int64_t n = host_hip::device_bytes;
    *planned = h->tiles.launches.size() == 1 && h->tiles.closed;
    xpbd_destroy(h);
    return n;
}

int main(int argc, char** argv)
{
    if (argc != 5) return 2;
    const Cube small(atoi(argv[1])), large(atoi(argv[3]));
    const int count = atoi(argv[2]);
    host_hip::units = atoi(argv[4]);
    for (int even = 0; even < 2; even++) {
        auto batch = [&](bool faces) {
            std::vector<xpbd_mesh_desc> d(even ? host_hip::units : count, (even ? large : small).desc(faces));
            if (!even) d.insert(d.begin() + d.size() / 2, large.desc(faces));
            return d;
        };
        bool planned = false, none = false;
        const int64_t plain = held(batch(false), XPBD_VARIANT_CLUSTER_QUAD, &none);
        const int64_t tiles = held(batch(false), XPBD_VARIANT_AUTO, &planned);
        const int64_t faces = held(batch(true), XPBD_VARIANT_CLUSTER_QUAD, &none);
        int64_t nv = 0;
        for (const auto& d : batch(false)) nv += d.num_vertices;
        printf("%lld %lld %d %lld\n", (long long)(tiles - plain), (long long)(faces - plain), (int)planned, (long long)nv);
    }
    return host_hip::device_bytes != 0;
}
