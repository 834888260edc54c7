// Plan of the vertex-tile Jacobi iteration (jacobi_tile_kernels.hip).
//
// Every vertex has an owner tile.  A tile projects all elements around its own
// vertices, those at its border as its neighbours do too, so that it alone forms
// its vertices' sums: one launch an iteration, with nothing to add up between
// tiles.  It reads the motions of all vertices of these elements from its own run
// of slots and writes its own vertices' to every slot that reads them.
#pragma once
#include <cstdint>
#include <vector>

namespace xpbd {

struct JacobiMesh {
    int nv, nt, nf;
    const int32_t* tets;    // 4 vertices an element, solver order
    const int32_t* faces;   // 4 ints a face slot: vertices, instance
    int patch_size;
    const std::vector<int32_t>& face_patch;   // per face slot; empty: contacts at the end
    const std::vector<int64_t>& v_off;   // vertices by instance (or by run of instances that are to be a tile)
    const std::vector<double>& rest;     // 3 a vertex
};

struct JacobiTiles {
    static constexpr int kHead = 12;
    enum { V0, NV, OWN, T0, NT, F0, NF, O0, NO, G0 };   // head: first and number of slots, own vertices (the first of
                                                        // the slots), elements, faces, out entries; first group
    int ntiles = 0;
    int verts = 0, tets = 0, slots = 0;   // most of a tile: slots read, elements, correction slots
    bool closed = true;                   // no tile reads another's vertices
    std::vector<int32_t> head;
    std::vector<int32_t> vert;       // slot -> vertex
    std::vector<uint16_t> local;     // per tile element: 4 vertices among the tile's slots, then the correction slot
                                     // of each, or 0xffff where another tile owns the vertex
    std::vector<int32_t> home;       // per tile element: 2 * solver position + whether this tile keeps its multipliers
    std::vector<int32_t> face;       // per tile face: 2 * face slot + as above, vertices 0 | 1 << 16, vertex 2 |
                                     // correction slot 0 << 16, slots 1 | 2 << 16
    std::vector<int32_t> group;      // per 64 own vertices: first correction slot of elements, of faces
    // per slot, of an own vertex: its elements' ends of partial sums (64 bits), which of these ends have contacts
    // to add (64), elements | faces << 16, its faces' ends of partial sums, 2 unused
    static constexpr int kSums = 8;
    std::vector<uint32_t> sums;
    std::vector<int32_t> out;        // own vertex, slot that reads it
    std::vector<int32_t> owner;      // vertex -> its owner's slot
};

// parts <= 0: a tile an instance.  threads: to build with.  False if a tile is too
// large for its 16-bit numbers, or a vertex has more than 64 elements or 32 faces.
bool build_jacobi_tiles(const JacobiMesh& M, int parts, int threads, JacobiTiles& J);

}  // namespace xpbd
