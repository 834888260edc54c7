// Builds a handle's fused-colour Gauss-Seidel plan: which colours share a
// launch, how many tiles a launch has, and the device data of each.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <exception>
#include <utility>

#include "capi_internal.h"
#include "gs_tile_kernels.h"
#include "gs_tiles.h"
#include "host_threads.h"
#include "pack.h"

using namespace xpbd;

namespace {

template <typename T>
int put(xpbd_handle* h, const T** dst, const std::vector<T>& v)
{
    void* p = nullptr;
    int rc = dalloc_bytes(h, &p, sizeof(T) * v.size());
    if (rc) return rc;
    if (!v.empty()) {
        hipError_t e = hipMemcpy(p, v.data(), sizeof(T) * v.size(), hipMemcpyHostToDevice);
        if (e != hipSuccess) return hip_err(h, e, "tile lists");
    }
    *dst = static_cast<const T*>(p);
    return XPBD_OK;
}

template <typename T>
int room(xpbd_handle* h, T** dst, size_t n)
{
    void* p = nullptr;
    int rc = dalloc_bytes(h, &p, sizeof(T) * n);
    *dst = static_cast<T*>(p);
    return rc;
}

int upload(xpbd_handle* h, const GsTileGroup& G, const GsTileDeal& deal, const GsTileShape& shape, GsTileLaunch& L)
{
    const int nblocks = G.ntiles * G.waves * G.blocks;
    const size_t rows = (size_t)G.ntiles * G.waves * G.rows, slots = (size_t)G.ntiles * G.slots;
    const int32_t *tile = nullptr, *wave = nullptr, *list = nullptr, *out = nullptr, *row = nullptr, *clu = nullptr;
    const uint8_t* own = nullptr;
    const uint16_t* vert = nullptr;
    float4* stream = nullptr;
    float2* lam = nullptr;
    int32_t* home = nullptr;
    int rc = put(h, &tile, G.tile);
    if (!rc) rc = put(h, &wave, G.wave);
    if (!rc) rc = put(h, &list, G.list);
    if (!rc) rc = put(h, &out, G.out);
    if (!rc) rc = put(h, &row, G.row);
    if (!rc) rc = put(h, &clu, G.clu);
    if (!rc) rc = put(h, &own, G.own);
    if (!rc) rc = put(h, &vert, G.vert);
    if (!rc && shape.lanes == 1) rc = room(h, &home, (size_t)nblocks * deal.per_block);
    if (!rc) rc = room(h, &stream, rows * (shape.lanes == 1 ? kLaneRow : 64));
    if (!rc) rc = room(h, &lam, rows * deal.per_block);
    if (!rc) rc = room(h, &L.d[0], slots);
    if (rc) return rc;
    hipError_t e = launch_fill_zero(h->stream, lam, sizeof(float2) * rows * deal.per_block);
    if (e == hipSuccess) e = launch_fill_zero(h->stream, L.d[0], sizeof(float4) * slots);
    if (e != hipSuccess) return hip_err(h, e, "tile set-up");
    GsTileFill F{};
    F.ta = tet_arrays(h);
    F.cstart = h->d_cstart;
    F.tloc = h->d_tloc;
    F.list = list;
    F.row = row;
    F.clu = clu;
    F.own = own;
    F.vert = vert;
    F.stream = stream;
    F.lam = lam;
    F.home = home;
    F.nblocks = nblocks;
    F.slots = G.slots;
    e = launch_gs_tile_fill(h->stream, F, shape);
    if (e != hipSuccess) return hip_err(h, e, "gs_tile_fill launch");
    GsTileArgs& A = L.args;
    A.tile = reinterpret_cast<const int2*>(tile);
    A.wave = reinterpret_cast<const int2*>(wave);
    A.list = list;
    A.out = reinterpret_cast<const int2*>(out);
    A.home = home;
    A.stream = stream;
    A.lam = lam;
    A.dlam = h->d_lam;
    A.waves = G.waves;
    A.slots = G.slots;
    A.rows = G.rows;
    A.blocks = G.blocks;
    A.outs = G.outs;
    A.nt = h->nt;
    L.nslots = (int)slots;
    L.ntiles = G.ntiles;
    L.smem = gs_tile_smem(G.slots, shape);
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
// 1,562 and 2,156).  Where a tile's phases or vertices do not fit (88^3), and above
// tp = 512, there is no plan.
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

// The groups of one try, on a thread each; false if memory ran out.
bool build_groups(const GsClusters& C, int nc, int m, int tp, bool whole, const GsTileDeal& deal,
                  std::vector<GsTileGroup>& G)
{
    G.assign((nc + m - 1) / m, GsTileGroup{});
    std::vector<char> bad(G.size(), 0);
    auto build = [&](size_t g) {
        try {
            const int c0 = (int)g * m, c1 = std::min(nc, c0 + m), n = C.color_off[c1] - C.color_off[c0];
            build_gs_tiles(C, c0, c1, whole ? 0 : (n + (c1 - c0) * tp - 1) / ((c1 - c0) * tp), deal, G[g]);
        } catch (const std::exception&) {
            bad[g] = 1;
        }
    };
    // threads pay for themselves on meshes that take a thread some milliseconds
    const size_t nthreads = C.color_off[nc] < 20000 ? 1 : std::min<size_t>(4, G.size());
    std::atomic<size_t> next{ 0 };
    on_threads(nthreads, [&] {
        for (size_t g; (g = next++) < G.size();) build(g);
    });
    return std::find(bad.begin(), bad.end(), 1) == bad.end();
}

int make_tiles(xpbd_handle* h)
{
    GsTilePlan& P = h->tiles;
    if (h->params.solver != XPBD_SOLVER_GS_COLORED || h->nclusters <= 0) return XPBD_OK;
    const int ncl = h->nclusters, nc = h->ncolors;
    int units = 0;
    hipError_t e = hipDeviceGetAttribute(&units, hipDeviceAttributeMultiprocessorCount, h->device);
    if (e != hipSuccess || units <= 0) return hip_err(h, e, "device attribute");
    int most = 0, whole_most = 0;   // clusters of a colour; of a colour and instance
    for (int c = 0; c < nc; c++) most = std::max(most, h->color_off[c + 1] - h->color_off[c]);
    const int tp = std::max(8, (most + units - 1) / units);
    std::vector<TileTry> tries;
    tile_tries(tp, tries);
    if (tries.empty()) return XPBD_OK;
    std::vector<int32_t> cverts(8 * (size_t)ncl), cinst(ncl, 0);
    e = hipMemcpy(cverts.data(), h->d_cverts, sizeof(int32_t) * cverts.size(), hipMemcpyDeviceToHost);
    if (e != hipSuccess) return hip_err(h, e, "cluster table");
    std::vector<float> centre(3 * (size_t)ncl);
    for (int i = 0; i < ncl; i++) {
        double s[3] = { 0, 0, 0 };
        int n = 0;
        for (int k = 0; k < 8; k++) {
            const int v = cverts[8 * (size_t)i + k];
            if (v < 0) continue;
            for (int a = 0; a < 3; a++) s[a] += h->rest[3 * (size_t)v + a];
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
    const GsClusters C{ h->nv, cverts, h->color_off, h->cl_start, cinst, centre };
    const int rows = h->cluster_max_tets <= 6 ? 6 : 8;
    const int whole_limit = nc > 16 ? 256 : 64;
    const bool whole = whole_most <= whole_limit && verts < 65535 &&
                       gs_tile_smem((int)verts + 1, GsTileShape{}) <= kGsTileLds;
    if (whole) {
        tries = { { nc, 4, 1 << 30, 1 << 20 } };
        pack_instances(h, units, whole_limit, cinst);
    }
    std::vector<GsTileGroup> G;
    GsTileDeal deal{};
    for (const TileTry& t : tries) {
        deal = t.lanes == 1 ? GsTileDeal{ 64, 8, rows, 0 } : GsTileDeal{ 16, 16, 0, 1 };
        if (!build_groups(C, nc, t.colours, tp, whole, deal, G)) return set_err(h, XPBD_E_NOMEM, "tile plan");
        int slots = 0, blocks = 0, least = rows;
        int64_t copies = 0;
        for (const GsTileGroup& g : G) {
            slots = std::max(slots, g.slots);
            blocks = std::max(blocks, g.max_phase_blocks);
            least = std::min(least, g.min_rows);
            copies += g.copies;
        }
        P.shape.lanes = t.lanes;
        P.shape.rows = rows;
        P.shape.full = least == 6;
        P.shape.cap = t.lanes == 1 ? gs_tile_cap(slots) : 0;
        const bool fits = slots <= 65535 && (t.lanes == 4 || P.shape.cap > 0) && gs_tile_smem(slots, P.shape) <= kGsTileLds;
        if (fits && blocks <= t.most_blocks && 10 * copies <= (int64_t)t.copies_tenths * ncl) break;
        G.clear();
    }
    if (G.empty()) return XPBD_OK;
    P.closed = G.size() == 1 && G[0].closed;
    // A solve first brings the bases into their slots.  With one iteration that is most of
    // what large one-lane plans gain (us a step, tiles and colour launches: tp = 140, 66^3, 111
    // and 121; 146, 300 cubes of 10^3, 119 and 123; 161, 700 objects, 139 and 122; 182, 72^3, 144
    // and 126; 250, 80^3, 165 and 151; with two iterations 239 and 232 at 72^3, 262 and 280 at 80^3).
    P.least = P.shape.lanes == 1 && tp > 150 ? 2 : 1;
    std::vector<int32_t> off, copy;
    for (size_t g = G.size(); g-- > 0;) {
        gs_tile_copies(h->nv, G[(g + 1) % G.size()], off, copy);
        link_gs_tiles(G[g], off, copy);
    }
    gs_tile_copies(h->nv, G[0], off, copy);
    std::vector<GsTileLaunch> launches(G.size());
    std::vector<int32_t> sv;
    for (size_t g = 0; g < G.size(); g++) {
        GsTileLaunch& L = launches[g];
        int rc = upload(h, G[g], deal, P.shape, L);
        if (rc) return rc;
        // waves that take no block help with the slots
        L.threads = 64 * std::max(G[g].waves, P.shape.lanes == 1 ? 8 : 4);
        sv.insert(sv.end(), G[g].slot_vert.begin(), G[g].slot_vert.end());
    }
    P.nslots = (int)sv.size();
    int rc = put(h, &P.slot_vert, sv);
    if (!rc) rc = room(h, &P.base, sv.size());
    for (size_t g = 0, at = 0; g < G.size() && !rc; at += launches[g].nslots, g++) launches[g].args.base = P.base + at;
    if (!rc) rc = put(h, &P.owner, G[0].owner);
    if (!rc) rc = put(h, &P.copy_off, off);
    if (!rc) rc = put(h, &P.copy, copy);
    if (!rc && !P.closed) rc = room(h, &P.kept, (size_t)h->nt);
    // one group that is not closed reads and writes its own slots: two arrays in turn
    if (!rc && G.size() == 1 && !P.closed) {
        rc = room(h, &launches[0].d[1], (size_t)launches[0].nslots);
        if (!rc) {
            e = launch_fill_zero(h->stream, launches[0].d[1], sizeof(float4) * (size_t)launches[0].nslots);
            if (e != hipSuccess) rc = hip_err(h, e, "tile set-up");
        }
    }
    if (rc) return rc;
    e = gs_tile_prepare(P.shape);
    if (e == hipSuccess) e = hipStreamSynchronize(h->stream);
    if (e != hipSuccess) return hip_err(h, e, "gs_tile set-up");
    P.launches = std::move(launches);
    return XPBD_OK;
}

}  // namespace

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
