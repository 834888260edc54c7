// Tiles for the fused-colour Gauss-Seidel kernels: one launch runs several
// consecutive colours.
//
// A group is a run of consecutive colours [c0, c1).  Its clusters are cut into
// spatial tiles, one workgroup each.  A tile owns the vertices whose last
// cluster of the group lies in it, and runs every cluster that these vertices
// depend on: with a cluster, for each of its vertices the cluster of the group
// that wrote it before.  Clusters near a tile's border therefore run in more
// than one tile, from the same inputs, with the same result.  Every copy of a
// cluster keeps its own multipliers (equal by construction).
//
// A group has its own array of in-step motions, a run of slots per tile with
// every vertex that the tile reads.  A launch reads its group's array and
// writes each owned vertex to all its slots of the next group's array, so no
// tile waits for another, what a tile reads is contiguous, and where its
// results go is known while it still computes.
//
// The result is that of projecting the group's clusters one by one in solver
// order: within a tile colours run in order, and clusters of one colour share
// no vertex.
#pragma once
#include <cstdint>
#include <vector>

namespace xpbd {

// How a tile's clusters are dealt to waves: a block is a wave's clusters of one
// phase (colour), one in each lane or each quad of lanes.
struct GsTileDeal {
    int per_block;    // clusters: 64 or 16
    int max_waves;    // of a workgroup that take blocks
    int pad_rows;     // element rows of every block, 0: as many as its largest cluster has
    int head_rows;    // rows before a block's element rows
};

struct GsTileGroup {
    int c0 = 0, c1 = 0;              // colours
    int ntiles = 0;
    int waves = 0;                   // that take blocks
    int slots = 0;                   // per tile: its vertices and, last, one that stands for none
    int rows = 0;                    // per tile and wave
    int blocks = 0;                  // per tile and wave
    int outs = 0;                    // per tile
    int min_rows = 16;               // fewest element rows of a block
    int max_phase_blocks = 0;        // most blocks of one phase of a tile
    int64_t copies = 0;              // clusters run, copies counted
    bool closed = false;             // no cluster runs in two tiles and no tile reads a vertex that it does not own
    std::vector<int32_t> tile;       // per tile (2): barriers an iteration (one ends a phase), entries of out
    std::vector<int32_t> wave;       // per tile and wave (2): blocks, barriers before the first
    std::vector<int32_t> list;       // per tile, wave and block: element rows | barriers until the wave's next << 4
    std::vector<int32_t> row;        // the block's first row (of all rows)
    std::vector<int32_t> clu;        // per block per_block solver clusters, -1 none
    std::vector<uint8_t> own;        // per cluster copy: it writes the multipliers back
    std::vector<uint16_t> vert;      // per cluster copy (8): tile slot of its vertices
    std::vector<int32_t> slot_vert;  // per tile and slot: vertex, -1 none
    std::vector<int32_t> owner;      // per vertex: the owner's slot, of all slots
    std::vector<int32_t> out;        // per tile (2 per entry): tile slot, slot of the next group
};

// cverts: 8 vertex ids per cluster in solver order (-1 padded); color_off:
// clusters of colour c are [color_off[c], color_off[c + 1]); cstart: first element
// of each cluster; cinst: instance of each cluster; centre: 3 floats per
// cluster.
struct GsClusters {
    int nv;
    const std::vector<int32_t>&cverts, &color_off, &cstart, &cinst;
    const std::vector<float>& centre;
    // lowest and highest vertex of each cluster along x, y, z (6 a cluster): where the same
    // plan is found sooner
    const std::vector<float>* extent = nullptr;
    int threads = 1;   // to cut with
};
// Cuts colours [c0, c1) into `parts` tiles (at most one per cluster), or with
// parts <= 0 makes every instance (every value of cinst) a tile.
void build_gs_tiles(const GsClusters& C, int c0, int c1, int parts, const GsTileDeal& deal, GsTileGroup& G);
// Slots of each vertex: copy[off[v] .. off[v + 1]).
void gs_tile_copies(int nv, const GsTileGroup& G, std::vector<int32_t>& off, std::vector<int32_t>& copy);
// Fills G.out: where each tile's owned vertices go in the next group, given its copies.
void link_gs_tiles(GsTileGroup& G, const std::vector<int32_t>& off, const std::vector<int32_t>& copy);

}  // namespace xpbd
