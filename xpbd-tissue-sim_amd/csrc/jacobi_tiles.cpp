#include "jacobi_tiles.h"

#include <algorithm>
#include <atomic>
#include <cstddef>
#include <exception>
#include <utility>

#include "host_threads.h"

namespace xpbd {

namespace {

// Cuts vertices [b, e) into parts of about equal size, instances apart first, then
// across the longest axis; tiles numbered from first on.
struct Cut {
    const JacobiMesh& M;
    std::vector<int32_t>& items;
    std::vector<int32_t>& tile;
    const std::vector<int32_t>& inst;
    std::vector<std::pair<double, int32_t>> key{};

    void run(int b, int e, int parts, int first)
    {
        if (parts <= 1 || e - b <= 1) {
            for (int i = b; i < e; i++) tile[items[i]] = first;
            return;
        }
        int lower = parts / 2, mid = b + (int)((int64_t)(e - b) * lower / parts);
        const auto mm = std::minmax_element(items.begin() + b, items.begin() + e);   // instances are runs of vertices
        if (inst[*mm.first] != inst[*mm.second]) {
            std::sort(items.begin() + b, items.begin() + e);
            int up = mid, dn = mid;
            while (up < e && inst[items[up]] == inst[items[up - 1]]) up++;
            while (dn > b && inst[items[dn]] == inst[items[dn - 1]]) dn--;
            mid = dn > b && (up >= e || mid - dn <= up - mid) ? dn : up;
            lower = (int)(((int64_t)parts * (mid - b) + (e - b) / 2) / (e - b));
            lower = std::min(parts - 1, std::max(1, lower));
        } else {
            double lo[3] = { 1e300, 1e300, 1e300 }, hi[3] = { -1e300, -1e300, -1e300 };
            for (int i = b; i < e; i++)
                for (int a = 0; a < 3; a++) {
                    const double x = M.rest[3 * (size_t)items[i] + a];
                    lo[a] = std::min(lo[a], x);
                    hi[a] = std::max(hi[a], x);
                }
            int axis = 0;
            for (int a = 1; a < 3; a++)
                if (hi[a] - lo[a] > hi[axis] - lo[axis]) axis = a;
            key.clear();   // by position and number
            for (int i = b; i < e; i++) key.emplace_back(M.rest[3 * (size_t)items[i] + axis], items[i]);
            std::nth_element(key.begin(), key.begin() + (mid - b), key.end());
            for (int i = b; i < e; i++) items[i] = key[i - b].second;
        }
        run(b, mid, lower, first);
        run(mid, e, parts - lower, first + lower);
    }
};

// items of each vertex: off, then ascending item numbers
void incidence(int nv, int n, int per, int stride, const int32_t* items, std::vector<int32_t>& off,
               std::vector<int32_t>& list)
{
    off.assign((size_t)nv + 1, 0);
    for (int i = 0; i < n; i++)
        for (int k = 0; k < per; k++) off[items[(size_t)stride * i + k] + 1]++;
    for (int v = 0; v < nv; v++) off[v + 1] += off[v];
    list.resize(off[nv]);
    std::vector<int32_t> at(off.begin(), off.end() - 1);
    for (int i = 0; i < n; i++)
        for (int k = 0; k < per; k++) list[at[items[(size_t)stride * i + k]]++] = i;
}

// One tile's lists, before its place among the others is known.
struct Tile {
    std::vector<int32_t> vert, home, face, group;
    std::vector<uint32_t> sums;
    std::vector<uint16_t> local;
    int own = 0, slots = 0;
    bool fits = true;
};

}  // namespace

bool build_jacobi_tiles(const JacobiMesh& M, int parts, int threads, JacobiTiles& J)
{
    const int nv = M.nv;
    J = JacobiTiles{};
    std::vector<int32_t> inst(nv, 0), tile(nv, 0);
    for (size_t i = 0; i + 1 < M.v_off.size(); i++)
        for (int64_t v = M.v_off[i]; v < M.v_off[i + 1]; v++) inst[v] = (int32_t)i;
    if (parts <= 0) {
        tile = inst;
        J.ntiles = (int)M.v_off.size() - 1;
    } else {
        J.ntiles = std::min(parts, std::max(1, nv));
        std::vector<int32_t> items(nv);
        for (int v = 0; v < nv; v++) items[v] = v;
        Cut{ M, items, tile, inst }.run(0, nv, J.ntiles, 0);
    }
    std::vector<int32_t> toff, tlist, foff, flist, own_off((size_t)J.ntiles + 1, 0), own(nv);
    incidence(nv, M.nt, 4, 4, M.tets, toff, tlist);
    incidence(nv, M.nf, 3, 4, M.faces, foff, flist);
    for (int v = 0; v < nv; v++) own_off[tile[v] + 1]++;
    for (int t = 0; t < J.ntiles; t++) own_off[t + 1] += own_off[t];
    {
        std::vector<int32_t> at(own_off.begin(), own_off.end() - 1);
        for (int v = 0; v < nv; v++) own[at[tile[v]]++] = v;
    }
    std::vector<Tile> tiles(J.ntiles);
    std::atomic<int> next{ 0 };
    std::atomic<bool> bad{ false };
    auto patch_of = [&](int face) { return M.face_patch.empty() ? 0 : M.face_patch[face]; };
    auto by_patch = [&](int f, int g) { return patch_of(f) != patch_of(g) ? patch_of(f) < patch_of(g) : f < g; };
    auto work = [&] {
        try {
            std::vector<int32_t> mine;
            std::vector<int32_t> seen(nv, -1), place(nv, 0), taken(M.nt, -1), used, elements, faces;
            for (int t; (t = next++) < J.ntiles && !bad;) {
                Tile& L = tiles[t];
                L.vert.assign(own.begin() + own_off[t], own.begin() + own_off[t + 1]);
                L.own = (int)L.vert.size();
                // vertices of like degree side by side: the 64 of a group are summed in step
                std::stable_sort(L.vert.begin(), L.vert.end(), [&](int p, int q) {
                    const int a = toff[p + 1] - toff[p], b = toff[q + 1] - toff[q];
                    return a != b ? a > b : foff[p + 1] - foff[p] > foff[q + 1] - foff[q];
                });
                elements.clear();
                faces.clear();
                for (int v : L.vert) {
                    for (int k = toff[v]; k < toff[v + 1]; k++)
                        if (taken[tlist[k]] != t) {
                            taken[tlist[k]] = t;
                            elements.push_back(tlist[k]);
                        }
                    faces.insert(faces.end(), flist.begin() + foff[v], flist.begin() + foff[v + 1]);
                }
                std::sort(elements.begin(), elements.end());
                std::sort(faces.begin(), faces.end(), by_patch);
                faces.erase(std::unique(faces.begin(), faces.end()), faces.end());
                for (int i = 0; i < L.own; i++) {
                    seen[L.vert[i]] = t;
                    place[L.vert[i]] = i;
                }
                auto at = [&](int v) {
                    if (seen[v] != t) {
                        seen[v] = t;
                        place[v] = (int)L.vert.size();
                        L.vert.push_back(v);
                    }
                    return place[v];
                };
                const int groups = (L.own + 63) / 64;
                L.sums.assign(JacobiTiles::kSums * (size_t)L.own, 0);
                L.group.assign(2 * (size_t)groups, 0);
                for (int g = 0; g < groups; g++) {
                    int td = 0, fd = 0;
                    for (int i = 64 * g; i < std::min(L.own, 64 * g + 64); i++) {
                        const int v = L.vert[i];
                        const int nt = toff[v + 1] - toff[v], nf = foff[v + 1] - foff[v];
                        td = std::max(td, nt);
                        fd = std::max(fd, nf);
                        if (nt > 64 || nf > 32) {
                            L.fits = false;
                            continue;
                        }
                        const int32_t* te = tlist.data() + toff[v];   // past the end for a last vertex without elements
                        mine.assign(flist.begin() + foff[v], flist.begin() + foff[v + 1]);
                        std::sort(mine.begin(), mine.end(), by_patch);
                        uint64_t end = 0, con = 0;
                        uint32_t fend = 0;
                        for (int k = 0; k < nt; k++) {
                            const int p = te[k] / M.patch_size;
                            if (k + 1 < nt && te[k + 1] / M.patch_size == p) continue;
                            end |= 1ull << k;
                            for (int f : mine)
                                if (!M.face_patch.empty() && patch_of(f) == p) con |= 1ull << k;
                        }
                        for (int k = 0; k < nf; k++)
                            if (k + 1 == nf || patch_of(mine[k + 1]) != patch_of(mine[k])) fend |= 1u << k;
                        uint32_t* q = &L.sums[JacobiTiles::kSums * (size_t)i];
                        q[0] = (uint32_t)end, q[1] = (uint32_t)(end >> 32);
                        q[2] = (uint32_t)con, q[3] = (uint32_t)(con >> 32);
                        q[4] = (uint32_t)nt | (uint32_t)nf << 16;
                        q[5] = fend;
                    }
                    L.group[2 * (size_t)g] = L.slots;
                    L.group[2 * (size_t)g + 1] = L.slots + 64 * td;
                    L.slots += 64 * (td + fd);
                }
                // corrections in the order of the items, vertex by vertex
                used.assign(2 * (size_t)L.own, 0);
                auto slot = [&](int v, int kind) {
                    if (tile[v] != t) return 0xffff;
                    const int i = place[v];
                    return L.group[2 * (size_t)(i / 64) + kind] + 64 * used[2 * (size_t)i + kind]++ + i % 64;
                };
                L.local.reserve(8 * elements.size());
                L.home.reserve(elements.size());
                L.face.reserve(4 * faces.size());
                for (int e : elements) {
                    const int32_t* v = M.tets + 4 * (size_t)e;
                    for (int k = 0; k < 4; k++) L.local.push_back((uint16_t)at(v[k]));
                    for (int k = 0; k < 4; k++) L.local.push_back((uint16_t)slot(v[k], 0));
                    L.home.push_back(2 * e + (tile[v[0]] == t ? 1 : 0));
                }
                for (int f : faces) {
                    const int32_t* v = M.faces + 4 * (size_t)f;
                    const int l[3] = { at(v[0]), at(v[1]), at(v[2]) };
                    const int s0 = slot(v[0], 1), s1 = slot(v[1], 1), s2 = slot(v[2], 1);
                    L.face.push_back(2 * f + (tile[v[0]] == t ? 1 : 0));
                    L.face.push_back(l[0] | l[1] << 16);
                    L.face.push_back((int32_t)((uint32_t)l[2] | (uint32_t)s0 << 16));
                    L.face.push_back((int32_t)((uint32_t)s1 | (uint32_t)s2 << 16));
                }
                L.fits = L.fits && L.vert.size() < 0x7fff && L.slots < 0xffff;
                if (!L.fits) bad = true;
            }
        } catch (const std::exception&) {
            bad = true;
        }
    };
    on_threads(std::min(threads, J.ntiles), work);
    if (bad) return false;
    // side by side
    J.owner.assign(nv, 0);
    std::vector<int32_t> copies((size_t)nv + 1, 0);
    size_t v0 = 0;
    for (const Tile& L : tiles) {
        for (int i = 0; i < L.own; i++) J.owner[L.vert[i]] = (int32_t)(v0 + i);
        for (int v : L.vert) copies[v + 1]++;
        v0 += L.vert.size();
    }
    for (int v = 0; v < nv; v++) copies[v + 1] += copies[v];
    std::vector<int32_t> slot_of(v0), at(copies.begin(), copies.end() - 1);
    v0 = 0;
    for (const Tile& L : tiles)
        for (int v : L.vert) slot_of[at[v]++] = (int32_t)v0++;
    size_t nt = 0, nout = 0;
    for (const Tile& L : tiles) {
        nt += L.home.size();
        nout += L.vert.size();   // an entry a slot that reads
    }
    J.vert.reserve(v0);
    J.sums.reserve(JacobiTiles::kSums * v0);
    J.local.reserve(8 * nt);
    J.home.reserve(nt);
    J.out.reserve(2 * nout);
    for (const Tile& L : tiles) {
        const int32_t base[JacobiTiles::kHead] = { (int32_t)J.vert.size(), (int32_t)L.vert.size(), L.own,
                                                   (int32_t)J.home.size(), (int32_t)L.home.size(),
                                                   (int32_t)(J.face.size() / 4), (int32_t)(L.face.size() / 4),
                                                   (int32_t)(J.out.size() / 2), 0, (int32_t)(J.group.size() / 2), 0, 0 };
        J.head.insert(J.head.end(), base, base + JacobiTiles::kHead);
        for (int i = 0; i < L.own; i++)
            for (int k = copies[L.vert[i]]; k < copies[L.vert[i] + 1]; k++) {
                J.out.push_back(i);
                J.out.push_back(slot_of[k]);
            }
        J.head[J.head.size() - JacobiTiles::kHead + JacobiTiles::NO] = (int32_t)(J.out.size() / 2) - base[JacobiTiles::O0];
        J.closed = J.closed && (int)L.vert.size() == L.own;
        J.verts = std::max(J.verts, (int)L.vert.size());
        J.tets = std::max(J.tets, (int)L.home.size());
        J.slots = std::max(J.slots, L.slots);
        J.vert.insert(J.vert.end(), L.vert.begin(), L.vert.end());
        J.local.insert(J.local.end(), L.local.begin(), L.local.end());
        J.home.insert(J.home.end(), L.home.begin(), L.home.end());
        J.face.insert(J.face.end(), L.face.begin(), L.face.end());
        J.group.insert(J.group.end(), L.group.begin(), L.group.end());
        J.sums.insert(J.sums.end(), L.sums.begin(), L.sums.end());
        J.sums.resize(JacobiTiles::kSums * J.vert.size(), 0);
    }
    return true;
}

}  // namespace xpbd
