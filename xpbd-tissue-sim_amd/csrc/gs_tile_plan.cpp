// Builds a handle's fused-colour Gauss-Seidel plan: which colours share a
// launch, how many tiles a launch has, and the device data of each.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <exception>
#include <memory>
#include <thread>
#include <utility>

#include "capi_internal.h"
#include "gs_tile_kernels.h"
#include "gs_tiles.h"
#include "host_threads.h"
#include "pack.h"
#include "plan_memory.h"

using namespace xpbd;

namespace {

// What a group's launch and its set-up take of the plan's memory.
struct GroupArrays {
    const int32_t *list = nullptr, *row = nullptr, *clu = nullptr;
    const int2 *tile = nullptr, *wave = nullptr, *out = nullptr;
    const uint8_t* own = nullptr;
    const uint16_t* vert = nullptr;
    float4* stream = nullptr;
    float2* lam = nullptr;
    int32_t* home = nullptr;
};

void reserve(PlanMemory& M, const GsTileGroup& G, const GsTileDeal& deal, const GsTileShape& shape, GroupArrays& A,
             GsTileLaunch& L)
{
    const size_t rows = (size_t)G.ntiles * G.waves * G.rows;
    L.nslots = G.ntiles * G.slots;
    M.put(&A.tile, G.tile);
    M.put(&A.wave, G.wave);
    M.put(&A.list, G.list);
    M.put(&A.out, G.out);
    M.put(&A.row, G.row);
    M.put(&A.clu, G.clu);
    M.put(&A.own, G.own);
    M.put(&A.vert, G.vert);
    if (shape.lanes == 1) M.room(&A.home, (size_t)G.ntiles * G.waves * G.blocks * deal.per_block);
    M.room(&A.stream, rows * (shape.lanes == 1 ? kLaneRow : 64));
    M.zeros(&A.lam, rows * deal.per_block);
    M.zeros(&L.d[0], (size_t)L.nslots);
}

int set_up(xpbd_handle* h, const GsTileGroup& G, const GsTileShape& shape, const GroupArrays& M, GsTileLaunch& L)
{
    GsTileFill F{};
    F.ta = tet_arrays(h);
    F.cstart = h->d_cstart;
    F.tloc = h->d_tloc;
    F.list = M.list;
    F.row = M.row;
    F.clu = M.clu;
    F.own = M.own;
    F.vert = M.vert;
    F.stream = M.stream;
    F.lam = M.lam;
    F.home = M.home;
    F.nblocks = G.ntiles * G.waves * G.blocks;
    F.slots = G.slots;
    hipError_t e = launch_gs_tile_fill(h->stream, F, shape);
    if (e != hipSuccess) return hip_err(h, e, "gs_tile_fill launch");
    GsTileArgs& A = L.args;
    A.tile = M.tile;
    A.wave = M.wave;
    A.list = M.list;
    A.out = M.out;
    A.home = M.home;
    A.stream = M.stream;
    A.lam = M.lam;
    A.dlam = h->d_lam;
    A.waves = G.waves;
    A.slots = G.slots;
    A.rows = G.rows;
    A.blocks = G.blocks;
    A.outs = G.outs;
    A.nt = h->nt;
    L.ntiles = G.ntiles;
    L.smem = gs_tile_smem(G.slots, shape);
    // waves that take no block help with the slots
    L.threads = 64 * std::max(G.waves, shape.lanes == 1 ? 8 : 4);
    return XPBD_OK;
}

// What to try, in order: colours a launch, and one lane a cluster or four.
struct TileTry {
    int colours, lanes, most_blocks, copies_tenths;
};

// One plan from the mesh's size.  P is the most clusters of a colour, tp = P over
// the compute units, the clusters of a colour that a tile owns when every unit
// has one workgroup: with more tiles than units the launch takes a second round
// for the rest (56^3 cells, one lane a cluster: 1.56 times as long with 400 tiles as
// with 256).
//
// whole: every instance a tile (or several, pack_instances), all colours in a launch, all iterations too while
// no contacts come between: few enough clusters that each SIMD of one unit has
// one wave (4^3 cells: 196 us against 381 us for colour launches, 8^3: 211
// against 407; 10^3, two waves each: 316, against 256 below), or many small
// colours, where copies would be most of the work (51 colours of 4,448 elements:
// 853 against 1,922).
//
// Four lanes a cluster have the shorter chain, one lane half the instructions for a
// cluster.  Up to tp = 65 a phase's chain counts (us a step of 10 iterations, four
// lanes and 2 colours a launch, against the best of one lane: 36^3 363 and 487, beam
// 200x20x20 476 and 506, 46^3 519 and 519, 50^3 549 and 549), above the instructions
// (56^3 679 and 611, 66^3 905 and 739).  More colours a launch save launches and cost
// copies: four while the colours are small (10^3 253, 2 colours 293; 16^3 255 and 291;
// level from 20^3 on, 302 and 305), three with one lane while a tile's fullest phase
// has a wave for each SIMD and no more (56^3 611, 2 colours 649; 66^3 805 and 739).
// Two launches' phases hold up to 8 blocks of 64 clusters, a wave each.  Where they
// fit they win (72^3 990, colour launches 1,085; 80^3 1,044 and 1,312; 96^3, tp = 432,
// 1,562 and 2,156).  Where a tile's phases or vertices do not fit (86^3 to 94^3, from
// 98^3 on), and above tp = 512, there is no plan.  All of this is from boxes of one
// object.
void tile_tries(int tp, std::vector<TileTry>& t)
{
    if (tp <= 11) t.push_back({ 4, 4, 16, 32 });
    if (tp <= 65) t.push_back({ 2, 4, 64, 22 });
    else if (tp <= 512) {
        if (tp <= 90) t.push_back({ 3, 1, 4, 22 });
        t.push_back({ 2, 1, 8, 22 });
    }
}

// Of a batch of more objects than units: several small objects a tile, as many tiles as
// units, none of them with more clusters of a colour than `most`.  With an object a tile
// the launch takes rounds of tiles that each leave a wave's lanes nearly empty, and all
// tiles are stored alike (gs_tiles.h), so that they take, and stage, the largest object's
// slots times their number.  us a step of 10 iterations with an object each, with colour
// launches, and packed: 3,000 cells 111, 66, 38; 20,000 cells 573, 98, 61; 2,000 cubes of
// 3^3 495, 507, 268; 10,000 cells and a cube of 8^3 516, 450, 211 (3.0 GB, packed 0.1).
// cinst: instance of each cluster, then its tile.
void pack_instances(const xpbd_handle* h, int units, int most, std::vector<int32_t>& cinst)
{
    if (h->ninst <= units) return;
    const int nc = h->ncolors;
    std::vector<int64_t> load((size_t)h->ninst * (nc + 1), 0), limit(nc + 1, most);
    limit[nc] = (h->nv + units - 1) / units;
    for (int i = 0; i < h->ninst; i++) load[(size_t)i * (nc + 1) + nc] = h->v_off[i + 1] - h->v_off[i];
    for (int c = 0; c < nc; c++)
        for (int i = h->color_off[c]; i < h->color_off[c + 1]; i++) load[(size_t)cinst[i] * (nc + 1) + c]++;
    const std::vector<int32_t> tile = pack_objects(h->ninst, load, limit);
    for (int32_t& i : cinst) i = tile[i];
}

constexpr int kThreadClusters = 300;   // a thread pays for itself from some 0.1 ms on

// work(0..n - 1), on threads if the mesh is worth it; false if memory ran out
template <typename Work>
bool each_group(size_t n, int clusters, const Work& work)
{
    std::atomic<bool> bad{ false };
    std::atomic<size_t> next{ 0 };
    on_threads(clusters < kThreadClusters ? 1 : std::min<size_t>(8, n), [&] {
        for (size_t g; (g = next++) < n;) {
            try {
                work(g);
            } catch (const std::exception&) {
                bad = true;
            }
        }
    });
    return !bad;
}

// The groups of one try; false if memory ran out.
bool build_groups(const GsClusters& C, int nc, int m, int tp, bool whole, const GsTileDeal& deal,
                  std::vector<GsTileGroup>& G)
{
    G.assign((nc + m - 1) / m, GsTileGroup{});
    return each_group(G.size(), C.color_off[nc], [&](size_t g) {
        const int c0 = (int)g * m, c1 = std::min(nc, c0 + m), n = C.color_off[c1] - C.color_off[c0];
        build_gs_tiles(C, c0, c1, whole ? 0 : (n + (c1 - c0) * tp - 1) / ((c1 - c0) * tp), deal, G[g]);
    });
}

// Links every group to the next; off, copy: the first group's slots by vertex.
bool link_groups(int nv, std::vector<GsTileGroup>& G, std::vector<int32_t>& off, std::vector<int32_t>& copy)
{
    return each_group(G.size(), nv, [&](size_t g) {
        std::vector<int32_t> o, c;
        gs_tile_copies(nv, G[(g + 1) % G.size()], o, c);
        link_gs_tiles(G[g], o, c);
        if (g + 1 < G.size()) return;
        off = std::move(o);
        copy = std::move(c);
    });
}

}  // namespace

// What a plan is on the host: all of it that takes no device memory.
struct xpbd::GsPlanHost {
    int units = 0;
    std::vector<int32_t> cverts;
    int rc = XPBD_OK;
    std::vector<GsTileGroup> G;   // empty where no plan fits
    GsTileDeal deal{};
    GsTileShape shape;
    bool closed = false;
    int least = 1;
    std::vector<int32_t> off, copy, slot_vert;   // off, copy: the first group's slots by vertex
    std::thread worker;
    ~GsPlanHost()
    {
        if (worker.joinable()) worker.join();
    }
};

namespace {

int plan_host(const xpbd_handle* h, GsPlanHost& H)
{
    const int units = H.units, ncl = h->nclusters, nc = h->ncolors;
    const std::vector<int32_t>& cverts = H.cverts;
    int most = 0, whole_most = 0;   // clusters of a colour; of a colour and instance
    for (int c = 0; c < nc; c++) most = std::max(most, h->color_off[c + 1] - h->color_off[c]);
    const int tp = std::max(8, (most + units - 1) / units);
    std::vector<TileTry> tries;
    tile_tries(tp, tries);
    if (tries.empty()) return XPBD_OK;
    std::vector<int32_t> cinst(ncl, 0);
    std::vector<float> centre(3 * (size_t)ncl), extent(6 * (size_t)ncl);
    for (int i = 0; i < ncl; i++) {
        double s[3] = { 0, 0, 0 };
        int n = 0;
        float* x = &extent[6 * (size_t)i];
        for (int a = 0; a < 3; a++) x[2 * a] = 1e30f, x[2 * a + 1] = -1e30f;
        for (int k = 0; k < 8; k++) {
            const int v = cverts[8 * (size_t)i + k];
            if (v < 0) continue;
            for (int a = 0; a < 3; a++) {
                const double r = h->rest[3 * (size_t)v + a];
                s[a] += r;
                x[2 * a] = std::min(x[2 * a], (float)r);
                x[2 * a + 1] = std::max(x[2 * a + 1], (float)r);
            }
            n++;
        }
        for (int a = 0; a < 3; a++) centre[3 * (size_t)i + a] = (float)(s[a] / n);
        if (h->ninst > 1)
            cinst[i] = (int32_t)(std::upper_bound(h->v_off.begin(), h->v_off.end(), (int64_t)cverts[8 * (size_t)i]) -
                                 h->v_off.begin()) - 1;
    }
    int64_t verts = 0;   // of an instance
    for (int i = 0; i < h->ninst; i++) verts = std::max(verts, h->v_off[i + 1] - h->v_off[i]);
    {
        std::vector<int32_t> n(h->ninst);
        for (int c = 0; c < nc; c++) {
            std::fill(n.begin(), n.end(), 0);
            for (int i = h->color_off[c]; i < h->color_off[c + 1]; i++) whole_most = std::max(whole_most, ++n[cinst[i]]);
        }
    }
    GsClusters C{ h->nv, cverts, h->color_off, h->cl_start, cinst, centre, &extent };
    const int rows = h->cluster_max_tets <= 6 ? 6 : 8;
    const int whole_limit = nc > 16 ? 256 : 64;
    const bool whole = whole_most <= whole_limit && verts < 65535 &&
                       gs_tile_smem((int)verts + 1, GsTileShape{}) <= kGsTileLds;
    if (whole) {
        tries = { { nc, 4, 1 << 30, 1 << 20 } };
        pack_instances(h, units, whole_limit, cinst);
    }
    std::vector<GsTileGroup>& G = H.G;
    GsTileDeal& deal = H.deal;
    for (const TileTry& t : tries) {
        deal = t.lanes == 1 ? GsTileDeal{ 64, 8, rows, 0 } : GsTileDeal{ 16, 16, 0, 1 };
        const int ngroups = (nc + t.colours - 1) / t.colours;
        C.threads = ncl < 8000 ? 1 : std::max(1, 8 / ngroups);   // smaller ones are cut in less than threads take
        if (!build_groups(C, nc, t.colours, tp, whole, deal, G)) return XPBD_E_NOMEM;
        int slots = 0, blocks = 0, least = rows;
        int64_t copies = 0;
        for (const GsTileGroup& g : G) {
            slots = std::max(slots, g.slots);
            blocks = std::max(blocks, g.max_phase_blocks);
            least = std::min(least, g.min_rows);
            copies += g.copies;
        }
        H.shape.lanes = t.lanes;
        H.shape.rows = rows;
        H.shape.full = least == 6;
        H.shape.cap = t.lanes == 1 ? gs_tile_cap(slots) : 0;
        const bool fits = slots <= 65535 && (t.lanes == 4 || H.shape.cap > 0) && gs_tile_smem(slots, H.shape) <= kGsTileLds;
        if (fits && blocks <= t.most_blocks && 10 * copies <= (int64_t)t.copies_tenths * ncl) break;
        G.clear();
    }
    if (G.empty()) return XPBD_OK;
    H.closed = G.size() == 1 && G[0].closed;
    // A solve first brings the bases into their slots.  With one iteration that is most of
    // what large one-lane plans gain (us a step, tiles and colour launches: tp = 140, 66^3, 111
    // and 121; 146, 300 cubes of 10^3, 119 and 123; 161, 700 objects, 139 and 122; 182, 72^3, 144
    // and 126; 250, 80^3, 165 and 151; with two iterations 239 and 232 at 72^3, 262 and 280 at 80^3).
    H.least = H.shape.lanes == 1 && tp > 150 ? 2 : 1;
    if (!link_groups(h->nv, G, H.off, H.copy)) return XPBD_E_NOMEM;
    for (const GsTileGroup& g : G) H.slot_vert.insert(H.slot_vert.end(), g.slot_vert.begin(), g.slot_vert.end());
    return XPBD_OK;
}

int plan_host_checked(const xpbd_handle* h, GsPlanHost& H)
{
    try {
        return plan_host(h, H);
    } catch (const std::exception&) {
        return XPBD_E_NOMEM;
    }
}

int make_tiles(xpbd_handle* h)
{
    GsTilePlan& P = h->tiles;
    if (h->params.solver != XPBD_SOLVER_GS_COLORED || h->nclusters <= 0) return XPBD_OK;
    std::shared_ptr<GsPlanHost> H = std::move(h->gs_begun);
    if (H) {
        H->worker.join();
    } else {
        H = std::make_shared<GsPlanHost>();
        int rc = device_units(h, &H->units);
        if (rc) return rc;
        H->cverts.resize(8 * (size_t)h->nclusters);
        hipError_t e = hipMemcpy(H->cverts.data(), h->d_cverts, sizeof(int32_t) * H->cverts.size(), hipMemcpyDeviceToHost);
        if (e != hipSuccess) return hip_err(h, e, "cluster table");
        H->rc = plan_host_checked(h, *H);
    }
    if (H->rc) return set_err(h, H->rc, "tile plan");
    const std::vector<GsTileGroup>& G = H->G;
    if (G.empty()) return XPBD_OK;
    P.shape = H->shape;
    P.closed = H->closed;
    P.least = H->least;
    std::vector<GsTileLaunch> launches(G.size());
    std::vector<GroupArrays> arrays(G.size());
    PlanMemory M;
    for (size_t g = 0; g < G.size(); g++) reserve(M, G[g], H->deal, P.shape, arrays[g], launches[g]);
    P.nslots = (int)H->slot_vert.size();
    M.put(&P.slot_vert, H->slot_vert);
    M.put(&P.owner, G[0].owner);
    M.put(&P.copy_off, H->off);
    M.put(&P.copy, H->copy);
    M.room(&P.base, H->slot_vert.size());
    if (!P.closed) M.room(&P.kept, (size_t)h->nt);
    // one group that is not closed reads and writes its own slots: two arrays in turn
    if (G.size() == 1 && !P.closed) M.zeros(&launches[0].d[1], (size_t)launches[0].nslots);
    int rc = M.place(h);
    for (size_t g = 0, at = 0; g < G.size() && !rc; at += launches[g].nslots, g++) {
        rc = set_up(h, G[g], P.shape, arrays[g], launches[g]);
        launches[g].args.base = P.base + at;
    }
    if (rc) return rc;
    hipError_t e = gs_tile_prepare(P.shape);
    if (e == hipSuccess) e = hipStreamSynchronize(h->stream);
    if (e != hipSuccess) return hip_err(h, e, "gs_tile set-up");
    P.launches = std::move(launches);
    return XPBD_OK;
}

}  // namespace

void xpbd::begin_gs_tiles(xpbd_handle* h, const std::vector<int32_t>& cluster_verts)
{
    if (h->nclusters < kThreadClusters) return;
    try {
        auto H = std::make_shared<GsPlanHost>();
        H->cverts = cluster_verts;
        if (device_units(h, &H->units)) return;
        H->worker = std::thread([h, p = H.get()] { p->rc = plan_host_checked(h, *p); });
        h->gs_begun = std::move(H);
    } catch (const std::exception&) {   // no thread, or no memory for one: planned when it is due
    }
}

int xpbd::ensure_gs_tiles(xpbd_handle* h)
{
    if (h->tiles.built) return XPBD_OK;
    const size_t kept = h->allocs.size();
    int rc;
    try {
        rc = make_tiles(h);
    } catch (const std::exception&) {   // host memory: a text that needs none
        rc = set_err(h, XPBD_E_NOMEM, "tile plan");
    }
    if (rc) {   // the handle goes on with its other launch shapes
        for (; h->allocs.size() > kept; h->allocs.pop_back()) (void)hipFree(h->allocs.back());
        h->tiles = GsTilePlan{};
        (void)hipGetLastError();
    }
    h->tiles.built = true;
    return rc;
}
