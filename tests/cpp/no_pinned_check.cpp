// A handle where no pinned memory can be had: it is created, and its state is read as
// ever.  Velocities are what the mesh says; positions are rest + ((base + low part) +
// in-step motion) in FP64 of records written here.
#include <cstdio>
#include <vector>

#include "capi_internal.h"
#include "host_hip.h"
#include "mesh_tools.h"

using namespace xpbd;

int main()
{
    host_hip::no_pinned = true;
    std::vector<std::vector<double>> x(2), v(2), m(2);
    std::vector<std::vector<int32_t>> t(2);
    std::vector<xpbd_mesh_desc> d(2);
    for (int i = 0; i < 2; i++) {
        const double o[3] = { 0.1, -0.2, 0.3 };
        grid_mesh(3 + 5 * i, 4, 2, 0.01, 0.02, 0.03, o, x[i], t[i]);
        const int nt = (int)(t[i].size() / 4);
        m[i].assign(2 * (size_t)nt, 1000.0);
        m[i].resize(3 * (size_t)nt, 0.4);
        for (size_t k = 0; k < x[i].size(); k++) v[i].push_back(0.25 * (double)(k % 7) - i);
        d[i] = {};
        d[i].num_vertices = (int)(x[i].size() / 3);
        d[i].num_tets = nt;
        d[i].x0 = x[i].data();
        d[i].v0 = v[i].data();
        d[i].tets = t[i].data();
        d[i].E = d[i].rho = m[i].data();
        d[i].nu = m[i].data() + 2 * nt;
    }
    xpbd_params p{};
    p.dt = 1e-3;
    p.iters = 1;
    xpbd_handle* h = nullptr;
    if (xpbd_batch_create(2, d.data(), &p, &h) != XPBD_OK) return printf("refused: %s\n", xpbd_last_error(nullptr)), 1;
    const size_t n = 3 * (size_t)h->nv;
    std::vector<double> want(n), wantv(n), got(n, -1.0), one(n, -1.0);
    std::vector<float> got32(n, -1.f);
    for (int i = 0; i < h->nv; i++) {
        float4 b = make_float4(1e-3f * i, -2e-3f * i, 0.5f, h->d_pos[2 * i].w), l = make_float4(3e-11f, 1e-10f * i, 0.f, 0.f);
        float4 e = make_float4(1e-6f, 0.f, 1e-5f * i, 0.f);
        h->d_pos[2 * i] = b;
        h->d_pos[2 * i + 1] = e;
        h->d_lo[i] = l;
        const double u[3] = { (double)b.x + l.x + e.x, (double)b.y + l.y + e.y, (double)b.z + l.z + e.z };
        for (int k = 0; k < 3; k++) want[3 * (size_t)i + k] = h->rest[3 * (size_t)i + k] + u[k];
    }
    for (int i = 0, at = 0; i < 2; i++)
        for (double c : v[i]) wantv[at++] = c;
    int64_t bad = xpbd_get_positions(h, got.data()) + xpbd_get_positions_f32(h, got32.data());
    for (size_t k = 0; k < n; k++) bad += (got[k] != want[k]) + (got32[k] != (float)want[k]);
    for (int i = 0; i < 2; i++) {
        bad += xpbd_batch_get_positions(h, i, one.data());
        const size_t from = 3 * (size_t)h->v_off[i], to = 3 * (size_t)h->v_off[i + 1];
        for (size_t k = from; k < to; k++) bad += one[k - from] != want[k];
    }
    bad += xpbd_get_velocities(h, got.data());
    for (size_t k = 0; k < n; k++) bad += got[k] != wantv[k];
    printf("%zu numbers, %lld wrong\n", n, (long long)bad);
    xpbd_destroy(h);
    return bad != 0 || host_hip::device_bytes != 0;
}
