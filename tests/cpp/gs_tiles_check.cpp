// Runs the fused-colour plan of a mesh on the CPU and compares it with the
// colour order.  Every projection is replaced by an integer hash of the
// cluster's vertices, so that any read of a value that is one projection too
// old or too new changes the result.
//   gs_tiles_check NX NY NZ INSTANCES COLOURS PARTS PER_BLOCK WAVES
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <vector>

#include "gs_tiles.h"
#include "mesh_tools.h"

using namespace xpbd;

static uint64_t mix(uint64_t h)
{
    h ^= h >> 31;
    h *= 0x9E3779B97F4A7C15ull;
    return h ^ (h >> 29);
}

int main(int argc, char** argv)
{
    if (argc != 9) return 2;
    const int nx = atoi(argv[1]), ny = atoi(argv[2]), nz = atoi(argv[3]), ninst = atoi(argv[4]);
    const int m = atoi(argv[5]), parts = atoi(argv[6]);
    std::vector<double> x;
    std::vector<int32_t> t, inst_of_vertex;
    for (int i = 0; i < ninst; i++) {   // instances of different sizes, all at the origin
        std::vector<double> xi;
        std::vector<int32_t> ti;
        const double o[3] = { 0, 0, 0 };
        grid_mesh(nx + i, ny, nz + 2 * i, 0.01, 0.01, 0.01, o, xi, ti);
        const int32_t v0 = (int32_t)(x.size() / 3);
        for (int32_t v : ti) t.push_back(v + v0);
        x.insert(x.end(), xi.begin(), xi.end());
        inst_of_vertex.resize(x.size() / 3, i);
    }
    const int nv = (int)(x.size() / 3), nt = (int)(t.size() / 4);
    std::vector<int32_t> cst, cv, col;
    std::vector<uint32_t> tl;
    const int ncl = build_clusters(nt, t.data(), cst, cv, tl);
    const int nc = greedy_color(nv, ncl, kClusterVerts, cv.data(), col);
    std::vector<int32_t> off(nc + 1, 0), order(ncl), cverts, cstart(1, 0), cinst(ncl);
    for (int c : col) off[c + 1]++;
    for (int c = 0; c < nc; c++) off[c + 1] += off[c];
    std::vector<int32_t> fill(off.begin(), off.end() - 1);
    for (int i = 0; i < ncl; i++) order[fill[col[i]]++] = i;
    std::vector<float> centre(3 * (size_t)ncl, 0.f);
    for (int i = 0; i < ncl; i++) {
        int n = 0;
        for (int k = 0; k < 8; k++) {
            const int v = cv[8 * (size_t)order[i] + k];
            cverts.push_back(v);
            if (v < 0) continue;
            n++;
            for (int a = 0; a < 3; a++) centre[3 * (size_t)i + a] += (float)x[3 * (size_t)v + a];
        }
        for (int a = 0; a < 3; a++) centre[3 * (size_t)i + a] /= (float)n;
        cstart.push_back(cstart.back() + cst[order[i] + 1] - cst[order[i]]);
        cinst[i] = inst_of_vertex[cverts[8 * (size_t)i]];
    }
    // one pass in colour order; lam counts a cluster's projections
    auto project = [&](int c, uint64_t** v, uint64_t& lam) {
        uint64_t h = mix((uint64_t)c + 77 * ++lam);
        for (int k = 0; k < 8; k++)
            if (v[k]) h = mix(h ^ *v[k]);
        for (int k = 0; k < 8; k++)
            if (v[k]) *v[k] = mix(h + k);
    };
    std::vector<uint64_t> ref(nv), lref(ncl, 0);
    for (int v = 0; v < nv; v++) ref[v] = mix(v + 1);
    const std::vector<uint64_t> start = ref;
    const int iters = 3;
    for (int it = 0; it < iters; it++)
        for (int c = 0; c < ncl; c++) {
            uint64_t* v[8];
            for (int k = 0; k < 8; k++) v[k] = cverts[8 * (size_t)c + k] < 0 ? nullptr : &ref[cverts[8 * (size_t)c + k]];
            project(c, v, lref[c]);
        }
    // the plan
    const GsClusters C{ nv, cverts, off, cstart, cinst, centre };
    const GsTileDeal deal{ atoi(argv[7]), atoi(argv[8]), 0, 1 };
    std::vector<GsTileGroup> G;
    for (int c0 = 0; c0 < nc; c0 += m) {
        G.emplace_back();
        build_gs_tiles(C, c0, c0 + m < nc ? c0 + m : nc, parts, deal, G.back());
    }
    std::vector<int32_t> coff, copy;
    for (size_t g = 0; g < G.size(); g++) {
        gs_tile_copies(nv, G[(g + 1) % G.size()], coff, copy);
        link_gs_tiles(G[g], coff, copy);
    }
    std::vector<std::vector<uint64_t>> d(G.size()), lam(G.size());
    for (size_t g = 0; g < G.size(); g++) {
        d[g].assign(G[g].slot_vert.size(), 0);
        lam[g].assign(G[g].clu.size(), 0);
    }
    for (size_t s = 0; s < d[0].size(); s++)
        if (G[0].slot_vert[s] >= 0) d[0][s] = start[G[0].slot_vert[s]];
    std::vector<uint64_t> lout(ncl, 0);
    for (int it = 0; it < iters; it++)
        for (size_t g = 0; g < G.size(); g++) {
            GsTileGroup& g0 = G[g];
            const std::vector<uint64_t> in = d[g];          // a launch reads the slots as they were
            std::vector<uint64_t>& to = d[(g + 1) % G.size()];
            std::vector<uint64_t> out = to;
            for (int tile = 0; tile < g0.ntiles; tile++) {
                std::vector<uint64_t> l(in.begin() + (size_t)tile * g0.slots, in.begin() + (size_t)(tile + 1) * g0.slots);
                // waves advance phase by phase: barrier p is passed when every wave has reached it
                const int barriers = g0.tile[2 * (size_t)tile];
                std::vector<int> at(g0.waves, 0), when(g0.waves, 0);
                for (int w = 0; w < g0.waves; w++) {
                    const size_t tw = (size_t)tile * g0.waves + w;
                    when[w] = g0.wave[2 * tw] ? g0.wave[2 * tw + 1] : barriers;
                }
                for (int p = 0; p < barriers; p++)
                    for (int w = g0.waves - 1; w >= 0; w--) {
                        const size_t tw = (size_t)tile * g0.waves + w;
                        while (when[w] == p) {
                            const size_t b = tw * g0.blocks + at[w]++;
                            when[w] += g0.list[b] >> 4;
                            for (int q = 0; q < deal.per_block; q++) {
                                const size_t i = b * deal.per_block + q;
                                const int c = g0.clu[i];
                                if (c < 0) continue;
                                if (cstart[c + 1] - cstart[c] > (g0.list[b] & 15)) return puts("rows"), 1;
                                uint64_t* v[8];
                                for (int k = 0; k < 8; k++)
                                    v[k] = cverts[8 * (size_t)c + k] < 0 ? nullptr : &l[g0.vert[8 * i + k]];
                                project(c, v, lam[g][i]);
                                if (g0.own[i]) lout[c] = lam[g][i];
                            }
                            if (at[w] == g0.wave[2 * tw]) break;
                        }
                    }
                for (int w = 0; w < g0.waves; w++)
                    if (when[w] != barriers) return puts("barriers"), 1;
                for (int k = 0; k < g0.tile[2 * (size_t)tile + 1]; k++) {
                    const int32_t* o = &g0.out[2 * ((size_t)tile * g0.outs + k)];
                    out[o[1]] = l[o[0]];
                }
            }
            to = out;
        }
    int64_t bad = 0;
    for (int v = 0; v < nv; v++) {
        bad += d[0][G[0].owner[v]] != ref[v];
    }
    for (size_t s = 0; s < d[0].size(); s++)   // every copy, not only the owner's
        if (G[0].slot_vert[s] >= 0) bad += d[0][s] != ref[G[0].slot_vert[s]];
    for (int c = 0; c < ncl; c++) bad += lout[c] != lref[c];
    int64_t copies = 0;
    bool closed = true;
    for (const GsTileGroup& g : G) {
        copies += g.copies;
        closed = closed && g.closed;
    }
    printf("%d colours, %zu groups, %d tiles, %.2f copies, closed %d, wrong %lld\n", nc, G.size(), G[0].ntiles,
           (double)copies / ncl, (int)closed, (long long)bad);
    return bad != 0;
}
