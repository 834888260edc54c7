#include "gs_tiles.h"

#include <algorithm>
#include <atomic>
#include <cstddef>
#include <cstring>
#include <exception>
#include <new>

#include "host_threads.h"

namespace xpbd {

namespace {

constexpr int kV = 8;  // vertices of a cluster

// Whole numbers in the order of finite floats: positions and numbers compare as one.
uint64_t ordered(float x)
{
    x += 0.f;   // one zero
    uint32_t u;
    std::memcpy(&u, &x, sizeof u);
    return u & 0x80000000u ? ~u : u | 0x80000000u;
}

// Cuts items[b, e) into `parts` parts of about equal size; tile numbers from
// first on.  Instances are cut apart first; within one, the cut goes across the
// axis that leaves the fewest vertices on both sides.
struct Bisect {
    struct Part {
        int b, e, parts, first;
    };
    const GsClusters& C;
    std::vector<int32_t>& items;
    std::vector<int32_t>& tile;   // per item's cluster - base
    const int base;
    std::vector<int32_t> mark = std::vector<int32_t>(C.nv, 0);   // per vertex: stamp of the last lower side that touched it
    int stamp = 0;
    std::vector<uint64_t> key{};

    // A vertex on both sides lies no higher than the lower side reaches and no lower
    // than the upper side does: clusters that end before that are passed over.
    int cut_size(int axis, int b, int mid, int e)
    {
        float low = 1e30f, high = -1e30f;   // lowest of the upper side, highest of the lower
        const float* ext = C.extent ? C.extent->data() + 2 * axis : nullptr;
        if (ext) {
            for (int i = b; i < mid; i++) high = std::max(high, ext[6 * (size_t)items[i] + 1]);
            for (int i = mid; i < e; i++) low = std::min(low, ext[6 * (size_t)items[i]]);
        }
        stamp++;
        for (int i = b; i < mid; i++) {
            if (ext && ext[6 * (size_t)items[i] + 1] < low) continue;
            for (int k = 0; k < kV; k++) {
                const int v = C.cverts[(size_t)kV * items[i] + k];
                if (v >= 0) mark[v] = stamp;
            }
        }
        int n = 0;
        for (int i = mid; i < e; i++) {
            if (ext && ext[6 * (size_t)items[i]] > high) continue;
            for (int k = 0; k < kV; k++) {
                const int v = C.cverts[(size_t)kV * items[i] + k];
                if (v >= 0) n += mark[v] == stamp;
            }
        }
        return n;
    }

    // items[b, e) with the lower ones along the axis in [b, mid), by position and number
    void along(int axis, int b, int mid, int e)
    {
        key.clear();
        for (int i = b; i < e; i++) key.push_back(ordered(C.centre[3 * (size_t)items[i] + axis]) << 32 | (uint32_t)items[i]);
        std::nth_element(key.begin(), key.begin() + (mid - b), key.end());
        for (int i = b; i < e; i++) items[i] = (int32_t)(key[i - b] & 0xffffffffu);
    }

    // Two parts of p, or false where it is one tile, which its items then have.
    bool split(const Part& p, Part& lo, Part& up)
    {
        const int b = p.b, e = p.e;
        if (p.parts <= 1 || e - b <= 1) {
            for (int i = b; i < e; i++) tile[items[i] - base] = p.first;
            return false;
        }
        const int lower = p.parts / 2;
        int mid = b + (int)((int64_t)(e - b) * lower / p.parts), lo_parts = lower;
        auto inst = [&](int i) { return C.cinst[items[i]]; };
        int32_t least = inst(b), most = least;
        for (int i = b; i < e; i++) {
            least = std::min(least, inst(i));
            most = std::max(most, inst(i));
        }
        if (least != most) {
            std::sort(items.begin() + b, items.begin() + e, [&](int x, int y) {
                return C.cinst[x] != C.cinst[y] ? C.cinst[x] < C.cinst[y] : x < y;
            });
            // the instance boundary nearest to the even cut, with parts in proportion
            int up = mid, dn = mid;
            while (up < e && inst(up) == inst(up - 1)) up++;
            while (dn > b && inst(dn) == inst(dn - 1)) dn--;
            mid = (dn > b && (up >= e || mid - dn <= up - mid)) ? dn : up;
            lo_parts = (int)(((int64_t)p.parts * (mid - b) + (e - b) / 2) / (e - b));
            lo_parts = std::min(p.parts - 1, std::max(1, lo_parts));
        } else {
            float lo[3], hi[3];
            for (int a = 0; a < 3; a++) lo[a] = 1e30f, hi[a] = -1e30f;
            for (int i = b; i < e; i++)
                for (int a = 0; a < 3; a++) {
                    lo[a] = std::min(lo[a], C.centre[3 * (size_t)items[i] + a]);
                    hi[a] = std::max(hi[a], C.centre[3 * (size_t)items[i] + a]);
                }
            int best = 0, best_cut = INT32_MAX, last = -1;
            for (int a = 0; a < 3; a++) {
                if (!(hi[a] > lo[a])) continue;
                along(a, b, mid, e);
                last = a;
                const int c = cut_size(a, b, mid, e);
                if (c < best_cut) best_cut = c, best = a;
            }
            if (last != best) along(best, b, mid, e);
        }
        lo = { b, mid, lo_parts, p.first };
        up = { mid, e, p.parts - lo_parts, p.first + lo_parts };
        return true;
    }

    void run(const Part& p)
    {
        Part lo, up;
        if (!split(p, lo, up)) return;
        run(lo);
        run(up);
    }
};

// All of items into parts: the first cuts one by one, what they leave on threads.
void bisect(const GsClusters& C, std::vector<int32_t>& items, std::vector<int32_t>& tile, int base, int parts)
{
    Bisect B{ C, items, tile, base };
    std::vector<Bisect::Part> left{ { 0, (int)items.size(), parts, 0 } };
    for (size_t i = 0; C.threads > 1 && i < left.size() && left.size() < 4 * (size_t)C.threads; i++) {
        Bisect::Part lo, up;   // breadth first: the largest parts are cut first
        const bool more = B.split(left[i], lo, up);
        left[i].parts = 0;   // done
        if (!more) continue;
        left.push_back(lo);
        left.push_back(up);
    }
    left.erase(std::remove_if(left.begin(), left.end(), [](const Bisect::Part& p) { return p.parts == 0; }), left.end());
    if (C.threads <= 1) {
        for (const Bisect::Part& p : left) B.run(p);
        return;
    }
    std::atomic<size_t> next{ 0 };
    std::atomic<bool> bad{ false };
    on_threads(C.threads, [&] {
        try {
            Bisect mine{ C, items, tile, base };
            for (size_t i; (i = next++) < left.size();) mine.run(left[i]);
        } catch (const std::exception&) {
            bad = true;
        }
    });
    if (bad) throw std::bad_alloc();
}

}  // namespace

void build_gs_tiles(const GsClusters& C, int c0, int c1, int parts, const GsTileDeal& deal, GsTileGroup& G)
{
    const auto &cverts = C.cverts, &color_off = C.color_off;
    const int nv = C.nv;
    G = GsTileGroup{};
    G.c0 = c0;
    G.c1 = c1;
    const int base = color_off[c0], n = color_off[c1] - base;
    const bool whole = parts <= 0;   // a tile an instance
    parts = whole ? 1 + *std::max_element(C.cinst.begin() + base, C.cinst.begin() + base + n) : std::min(parts, n);
    std::vector<int32_t> items(n), ctile(n, 0), color(n);
    for (int i = 0; i < n; i++) items[i] = base + i;
    for (int c = c0; c < c1; c++)
        for (int i = color_off[c]; i < color_off[c + 1]; i++) color[i - base] = c - c0;
    if (whole) {
        for (int i = 0; i < n; i++) ctile[i] = C.cinst[base + i];
    } else {
        bisect(C, items, ctile, base, parts);
    }
    G.ntiles = parts;
    // per vertex the last cluster of the group that touches it; per cluster and
    // vertex the one before it
    std::vector<int32_t> last(nv, -1), prev((size_t)kV * n, -1);
    for (int i = 0; i < n; i++)
        for (int k = 0; k < kV; k++) {
            const int v = cverts[(size_t)kV * (base + i) + k];
            if (v < 0) continue;
            prev[(size_t)kV * i + k] = last[v];
            last[v] = i;
        }
    // owner tile of every vertex; the untouched ones are spread over the tiles in index order
    std::vector<int32_t> owner(nv), oc(parts + 1, 0);
    int64_t untouched = 0, at = 0;
    for (int v = 0; v < nv; v++) untouched += last[v] < 0;
    for (int v = 0; v < nv; v++) {
        owner[v] = last[v] >= 0 ? ctile[last[v]] : (int)(at++ * parts / std::max<int64_t>(untouched, 1));
        oc[owner[v] + 1]++;
    }
    for (int t = 0; t < parts; t++) oc[t + 1] += oc[t];
    std::vector<int32_t> owned(nv), fill(oc.begin(), oc.end() - 1);
    for (int v = 0; v < nv; v++) owned[fill[owner[v]]++] = v;

    auto tets = [&](int i) { return C.cstart[base + i + 1] - C.cstart[base + i]; };
    const int nph = c1 - c0;
    std::vector<int32_t> seen(n, -1), vseen(nv, -1), stack, mine;
    std::vector<uint8_t> written(n, 0);
    // tile by tile: its clusters phase by phase, and its vertices in slot order
    std::vector<int32_t> run, roff{ 0 }, verts, voff{ 0 };
    std::vector<std::vector<int32_t>> by_phase(nph);
    G.closed = true;
    for (int t = 0; t < parts; t++) {
        mine.clear();
        auto need = [&](int i) {
            if (i >= 0 && seen[i] != t) {
                seen[i] = t;
                stack.push_back(i);
            }
        };
        for (int q = oc[t]; q < oc[t + 1]; q++) need(last[owned[q]]);
        while (!stack.empty()) {
            const int i = stack.back();
            stack.pop_back();
            mine.push_back(i);
            for (int k = 0; k < kV; k++) need(prev[(size_t)kV * i + k]);
        }
        std::sort(mine.begin(), mine.end());   // solver order
        for (auto& L : by_phase) L.clear();
        for (int i : mine) by_phase[color[i]].push_back(i);
        // a block has as many element rows as its largest cluster: clusters of like size together
        for (auto& L : by_phase) std::stable_sort(L.begin(), L.end(), [&](int x, int y) { return tets(x) > tets(y); });
        // Slots as the first phases' waves read them, vertex by vertex over the
        // clusters: neighbouring lanes then read neighbouring LDS words.
        for (const auto& L : by_phase)
            for (int k = 0; k < kV; k++)
                for (int i : L) {
                    const int v = cverts[(size_t)kV * (base + i) + k];
                    if (v >= 0 && vseen[v] != t) {
                        vseen[v] = t;
                        verts.push_back(v);
                        G.closed = G.closed && owner[v] == t;
                    }
                }
        for (int q = oc[t]; q < oc[t + 1]; q++)
            if (vseen[owned[q]] != t) {
                vseen[owned[q]] = t;
                verts.push_back(owned[q]);
            }
        voff.push_back((int32_t)verts.size());
        G.slots = std::max(G.slots, voff[t + 1] - voff[t] + 1);
        G.copies += (int64_t)mine.size();
        for (const auto& L : by_phase) {
            run.insert(run.end(), L.begin(), L.end());
            roff.push_back((int32_t)run.size());
            G.max_phase_blocks = std::max(G.max_phase_blocks, ((int)L.size() + deal.per_block - 1) / deal.per_block);
        }
    }
    // The phases' blocks dealt to the waves in turn, a phase's first to the wave
    // after the one that took the last phase's last.
    G.waves = std::min(deal.max_waves, std::max(1, G.max_phase_blocks));
    struct Block {
        int first, count, rows, phase;   // of run
    };
    std::vector<std::vector<Block>> wl((size_t)parts * G.waves);
    G.tile.assign(2 * (size_t)parts, 0);
    for (int t = 0; t < parts; t++) {
        int ph = 0, w = 0;   // phases without clusters take no barrier
        for (int p = 0; p < nph; p++) {
            const int r0 = roff[(size_t)t * nph + p], r1 = roff[(size_t)t * nph + p + 1];
            for (int r = r0; r < r1; r += deal.per_block, w = (w + 1) % G.waves) {
                const int rows = deal.pad_rows > 0 ? deal.pad_rows : tets(run[r]);
                G.min_rows = std::min(G.min_rows, rows);
                wl[(size_t)t * G.waves + w].push_back({ r, std::min(deal.per_block, r1 - r), rows, ph });
            }
            ph += r1 > r0;
        }
        G.tile[2 * (size_t)t] = ph;
        for (int w = 0; w < G.waves; w++) {
            const auto& L = wl[(size_t)t * G.waves + w];
            int rows = 0;
            for (const Block& b : L) rows += deal.head_rows + b.rows;
            G.rows = std::max(G.rows, rows);
            G.blocks = std::max(G.blocks, (int)L.size());
        }
    }
    G.blocks = std::max(G.blocks, 1);
    G.rows = std::max(G.rows, deal.head_rows + std::max(deal.pad_rows, kV));   // what a wave loads unasked
    const size_t nblk = wl.size() * G.blocks;
    G.wave.assign(2 * wl.size(), 0);
    G.list.assign(nblk, 0);
    G.row.assign(nblk, 0);
    G.clu.assign(nblk * deal.per_block, -1);
    G.own.assign(nblk * deal.per_block, 0);
    G.vert.assign(nblk * deal.per_block * kV, (uint16_t)(G.slots - 1));
    G.slot_vert.assign((size_t)parts * G.slots, -1);
    G.owner.assign(nv, -1);
    std::vector<int32_t> vlocal(nv, 0);
    for (int t = 0; t < parts; t++) {
        for (int q = voff[t]; q < voff[t + 1]; q++) {
            const int v = verts[q], s = q - voff[t];
            vlocal[v] = s;
            G.slot_vert[(size_t)t * G.slots + s] = v;
            if (owner[v] == t) G.owner[v] = t * G.slots + s;
        }
        for (int w = 0; w < G.waves; w++) {
            const size_t tw = (size_t)t * G.waves + w;
            const auto& L = wl[tw];
            G.wave[2 * tw] = (int32_t)L.size();
            G.wave[2 * tw + 1] = L.empty() ? 0 : L[0].phase;
            int row = (int)tw * G.rows;
            for (size_t i = 0; i < L.size(); i++) {
                const size_t b = tw * G.blocks + i;
                const int next = i + 1 < L.size() ? L[i + 1].phase : G.tile[2 * (size_t)t];
                G.list[b] = L[i].rows | (next - L[i].phase) << 4;
                G.row[b] = row;
                row += deal.head_rows + L[i].rows;
                for (int q = 0; q < L[i].count; q++) {
                    const int c = run[L[i].first + q];
                    const size_t at = b * deal.per_block + q;
                    G.clu[at] = base + c;
                    G.own[at] = !written[c];
                    if (written[c]) G.closed = false;
                    written[c] = 1;
                    for (int k = 0; k < kV; k++) {
                        const int v = cverts[(size_t)kV * (base + c) + k];
                        if (v >= 0) G.vert[at * kV + k] = (uint16_t)vlocal[v];
                    }
                }
            }
        }
    }
}

void gs_tile_copies(int nv, const GsTileGroup& G, std::vector<int32_t>& off, std::vector<int32_t>& copy)
{
    off.assign((size_t)nv + 1, 0);
    for (int v : G.slot_vert)
        if (v >= 0) off[v + 1]++;
    for (int v = 0; v < nv; v++) off[v + 1] += off[v];
    copy.resize(off[nv]);
    std::vector<int32_t> fill(off.begin(), off.end() - 1);
    for (size_t s = 0; s < G.slot_vert.size(); s++)
        if (G.slot_vert[s] >= 0) copy[fill[G.slot_vert[s]]++] = (int32_t)s;
}

void link_gs_tiles(GsTileGroup& G, const std::vector<int32_t>& off, const std::vector<int32_t>& copy)
{
    G.outs = 0;
    for (int pass = 0; pass < 2; pass++) {   // the longest list first, then the lists
        if (pass) G.out.assign(2 * (size_t)G.ntiles * std::max(G.outs, 1), 0);
        for (int t = 0; t < G.ntiles; t++) {
            int n = 0;
            for (int s = 0; s < G.slots; s++) {
                const int at = t * G.slots + s, v = G.slot_vert[at];
                if (v < 0 || G.owner[v] != at) continue;
                for (int k = off[v]; k < off[v + 1]; k++, n++)
                    if (pass) {
                        G.out[2 * ((size_t)t * G.outs + n)] = s;
                        G.out[2 * ((size_t)t * G.outs + n) + 1] = copy[k];
                    }
            }
            G.tile[2 * (size_t)t + 1] = n;
            if (!pass) G.outs = std::max(G.outs, n);
        }
    }
}

}  // namespace xpbd
