// Builds a handle's vertex-tile Jacobi plan: how many tiles, and the device data.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <exception>
#include <memory>
#include <thread>

#include "capi_internal.h"
#include "jacobi_tile_kernels.h"
#include "jacobi_tiles.h"
#include "pack.h"
#include "plan_memory.h"

using namespace xpbd;

namespace {

constexpr size_t kLds = 160 * 1024;   // of a workgroup, gfx950
constexpr int kThreadElements = 2000;   // a thread pays for itself from some 0.1 ms on

// Tiles of a plan, 0 for a tile an instance (or several, packed), -1 for no plan.  us a step of 10 iterations against the
// patch launches:
// - an instance a tile, all iterations in a launch, while an instance's elements are
//   one a thread: 4^3 cells 33 against 61 (tiles of few vertices: 57), 5^3 39 against
//   65; 6^3 is more, a tile 57 either way.
// - else a tile a compute unit, which is all that fit side by side: 12^3 56 against
//   75, 24^3 67 against 103, 40^3 147 against 167, beam 200x20x20 172 against 195.
//   Of fewer than 12 vertices a tile is mostly border (12^3 with 9: 59).
// A tile's corrections have to fit in LDS, up to some 400 vertices.  With more tiles
// than units the border's extra elements and the second round take what is gained
// (50^3: 246 against 246, 56^3 306 against 297): no plan.
int tile_count(const xpbd_handle* h, int units)
{
    int64_t most = 0;   // elements of an instance
    for (int i = 0; i < h->ninst; i++) most = std::max(most, h->t_off[i + 1] - h->t_off[i]);
    if (most <= 1024) return 0;
    const int own = std::max(12, (h->nv + units - 1) / units);
    if (own > 420) return -1;
    return (h->nv + own - 1) / own;
}

// Where an instance is a tile: the first vertex of each tile, and the end.  Of a batch
// of more objects than units several small ones share a tile, as many tiles as units, of
// at most an element a thread and 2,048 vertices (their records and corrections take
// 88 KB of LDS).  us a step of 10 iterations with an object each, with the patch
// launches, and packed: 20,000 cells 157, 102, 63; 2,000 cubes of 2^3 (48 elements) 74,
// 90, 49; 700 of 1..5 cells per axis (162 and 750) 76, 97, 61.  Objects that fill a wave and
// are alike gain nothing: 600 cubes of 3^3 39, 90, 43; 2,000 of them 72, 131, 85.
std::vector<int64_t> packed(const xpbd_handle* h, int units)
{
    std::vector<int64_t> load, v_off;
    int64_t most = 0;   // elements of an object
    for (int i = 0; i < h->ninst; i++) {
        load.push_back(h->t_off[i + 1] - h->t_off[i]);
        load.push_back(h->v_off[i + 1] - h->v_off[i]);
        most = std::max(most, load[2 * (size_t)i]);
    }
    if (h->ninst <= units || (h->nt >= 64ll * h->ninst && h->ninst * most <= 3ll * h->nt)) return h->v_off;
    const std::vector<int32_t> tile =
        pack_objects(h->ninst, load, { 1024, std::min<int64_t>(2048, (h->nv + units - 1) / units) });
    for (int i = 0; i < h->ninst; i++)
        if (i == 0 || tile[i] != tile[i - 1]) v_off.push_back(h->v_off[i]);
    v_off.push_back(h->nv);
    return v_off;
}

}  // namespace

// What a plan is on the host.
struct xpbd::JacobiPlanHost {
    int units = 0;
    std::vector<int32_t> faces;
    int rc = XPBD_OK;
    bool fits = false;
    JacobiTiles J;
    std::thread worker;
    ~JacobiPlanHost()
    {
        if (worker.joinable()) worker.join();
    }
};

namespace {

int plan_host(const xpbd_handle* h, JacobiPlanHost& H)
{
    try {
        const int parts = tile_count(h, H.units);
        if (parts < 0) return XPBD_OK;
        std::vector<int32_t> tets;
        tets.reserve(4 * (size_t)h->nt);
        for (int32_t t : h->order) {
            const int32_t* v = h->tets_host.data() + 4 * (size_t)t;
            tets.insert(tets.end(), v, v + 4);
        }
        const std::vector<int64_t> v_off = parts == 0 ? packed(h, H.units) : h->v_off;
        const JacobiMesh M{ h->nv, h->nt, h->nf, tets.data(), H.faces.data(), jacobi_patch_size(), h->face_patch, v_off, h->rest };
        const int threads = h->nt < kThreadElements ? 1 : h->nt < 8000 ? 4 : 8;
        H.fits = build_jacobi_tiles(M, parts, threads, H.J) && jacobi_tile_smem(H.J.verts, H.J.slots) <= kLds;
        return XPBD_OK;
    } catch (const std::exception&) {
        return XPBD_E_NOMEM;
    }
}

bool plannable(const xpbd_handle* h)
{
    return h->variant == XPBD_VARIANT_PATCH && h->params.deterministic != 0 && h->nt > 0;
}

int make_tiles(xpbd_handle* h)
{
    JacobiTilePlan& P = h->jtiles;
    if (!plannable(h)) return XPBD_OK;
    std::shared_ptr<JacobiPlanHost> H = std::move(h->jacobi_begun);
    if (H) {
        H->worker.join();
    } else {
        H = std::make_shared<JacobiPlanHost>();
        int rc = device_units(h, &H->units);
        if (rc) return rc;
        H->faces.resize(4 * (size_t)h->nf);
        if (h->nf > 0) {
            hipError_t e = hipMemcpy(H->faces.data(), h->d_faces, sizeof(int32_t) * H->faces.size(), hipMemcpyDeviceToHost);
            if (e != hipSuccess) return hip_err(h, e, "face table");
        }
        H->rc = plan_host(h, *H);
    }
    if (H->rc) return set_err(h, H->rc, "tile plan");
    if (!H->fits) return XPBD_OK;
    const JacobiTiles& J = H->J;
    JacobiTileArgs A{};
    const size_t n = J.home.size(), slots = J.vert.size();
    float4* stream = nullptr;
    float4* base = nullptr;
    PlanMemory memory;
    memory.put(&A.head, J.head);
    memory.put(&A.local, J.local);
    memory.put(&A.home, J.home);
    memory.put(&A.face, J.face);
    memory.put(&A.group, J.group);
    memory.put(&A.sums, J.sums);
    memory.put(&A.out, J.out);
    memory.put(&A.vert, J.vert);
    memory.put(&P.owner, J.owner);
    memory.room(&stream, 3 * n);
    memory.zeros(&A.lam, n);
    memory.room(&base, slots);
    for (float4*& d : P.d) memory.zeros(&d, slots);
    if (!J.closed) memory.room(&P.kept, (size_t)h->nt);
    int rc = memory.place(h);
    if (rc) return rc;
    hipError_t e = launch_jacobi_tile_fill(h->stream, tet_arrays(h), A.home, (int)n, stream);
    if (e == hipSuccess) e = jacobi_tile_prepare();
    if (e == hipSuccess) e = hipStreamSynchronize(h->stream);
    if (e != hipSuccess) return hip_err(h, e, "Jacobi tile set-up");
    A.stream = stream;
    A.base = base;
    A.dlam = h->d_lam;
    A.n = (int)n;
    A.verts = J.verts;
    A.slots = J.slots;
    A.ntiles = J.ntiles;
    A.late = h->face_patch.empty();
    A.flag = h->d_flag;
    A.rest = h->d_rest;
    A.lo = h->d_lo;
    A.cp = h->d_cp;
    A.cn = h->d_cn;
    A.cb = h->d_cb;
    A.clam = h->d_clam;
    P.args = A;
    P.base = base;
    P.closed = J.closed;
    P.nslots = (int)slots;
    P.threads = std::min(1024, std::max(64, (J.tets + 63) / 64 * 64));
    P.ready = true;
    return XPBD_OK;
}

}  // namespace

void xpbd::begin_jacobi_tiles(xpbd_handle* h, const int32_t* faces)
{
    if (!plannable(h) || h->nt < kThreadElements) return;
    try {
        auto H = std::make_shared<JacobiPlanHost>();
        H->faces.assign(faces, faces + 4 * (size_t)h->nf);
        if (device_units(h, &H->units)) return;
        H->worker = std::thread([h, p = H.get()] { p->rc = plan_host(h, *p); });
        h->jacobi_begun = std::move(H);
    } catch (const std::exception&) {   // no thread, or no memory for one: planned when it is due
    }
}

int xpbd::ensure_jacobi_tiles(xpbd_handle* h)
{
    if (h->jtiles.built) return XPBD_OK;
    const size_t kept = h->allocs.size();
    int rc;
    try {
        rc = make_tiles(h);
    } catch (const std::exception&) {   // host memory: a text that needs none
        rc = set_err(h, XPBD_E_NOMEM, "tile plan");
    }
    if (rc) {   // the handle goes on with its other launch shapes
        for (; h->allocs.size() > kept; h->allocs.pop_back()) (void)hipFree(h->allocs.back());
        h->jtiles = JacobiTilePlan{};
        (void)hipGetLastError();
    }
    h->jtiles.built = true;
    return rc;
}
