// plx_plan.hpp -- host-side tile plan (see plx_plan.cpp).
#pragma once

#include <algorithm>
#include <cmath>
#include <cstdint>
#include <string>
#include <vector>

namespace plx {

// Per-tile bounds that size the LDS of the cell kernels.
struct TileLimits {
    int cells;   // cells per tile = threads per workgroup
    int nodes;   // max distinct nodes per tile
    int verts;   // max distinct vertices per tile
};

inline TileLimits tile_limits(int cell_type) {
    if (cell_type == 1) return {512, 768, 768};  // Q1 hex: an 8^3 brick touches 729 nodes
    return {384, 768, 192};                      // P2 tet: 4^3 cubes x 6 touch 729 nodes
}

// Read-only view of the mesh arrays a plan is built from.
struct MeshView {
    int nb, nv;
    int num_cells, num_nodes, num_vertices;
    const int32_t *closure;
    const int32_t *cone;
    const int32_t *labels;  // may be null (all 0)
    bool cone_is_closure;   // isoparametric Q1: vertices are the nodes, in closure order
    const double *coords = nullptr;  // [num_vertices][3] (spatial reordering of badly ordered keys)
};

// Powers of two that keep the FP32 element of P2 tetrahedra in range (p2_geometry): area, near the inverse of a typical
// cell's squared length, for the adjugate of J, and its inverse square for the scale of the stresses.
struct P2Scale {
    float area = 1.0f;
    double factor = 1.0;
};
inline P2Scale p2_scale(const double *coords, int64_t num_vertices, int64_t num_cells) {
    double lo[3] = {1e300, 1e300, 1e300}, hi[3] = {-1e300, -1e300, -1e300}, size = 0.0;
    for (int64_t i = 0; i < num_vertices; ++i)
        for (int d = 0; d < 3; ++d) {
            lo[d] = std::min(lo[d], coords[3 * i + d]);
            hi[d] = std::max(hi[d], coords[3 * i + d]);
        }
    for (int d = 0; d < 3; ++d) size = std::max(size, hi[d] - lo[d]);
    const double length = size / std::cbrt((double)num_cells);
    if (!(length > 0.0) || !std::isfinite(length)) return P2Scale();
    const int e = std::max(-120, std::min(120, 2 * std::ilogb(length)));
    return {(float)std::ldexp(1.0, -e), std::ldexp(1.0, 2 * e)};
}

struct HostPlan {
    int num_tiles = 0;
    int max_nodes = 0, max_verts = 0, max_colors = 0;
    int64_t halo_slots = 0;
    std::vector<int32_t> cells;  // key cells in tile order
    std::vector<int32_t> tile_cell_ptr, tile_node_ptr, tile_nown, tile_nodes, tile_vert_ptr,
        tile_verts, tile_halo_off, tile_ncolor;
    std::vector<uint16_t> lclosure, lcone;  // [nb][ncells], [nv][ncells]
    std::vector<uint8_t> color;             // [ncells]
    // With cone_is_closure the vertex list of a tile IS its node list (same order), so the
    // kernels index staged coordinates with the local node index.
    std::vector<int32_t> shared_node, shared_ptr, shared_slot;
    bool reordered = false;  // cells taken in Morton order of their centroids instead of input order
};

// Tile plan of the P2 pair kernel: the key's cells in tiles of up to kPairTilePairs pairs of cells
// that share a face (a pair has 14 distinct nodes and 5 vertices where two cells have 20 and 8), one
// pair per thread.  A cell left without a partner is paired with its own mirror image, whose
// moduli the kernel reads as zero.
constexpr int kPairTilePairs = 256, kPairTileNodes = 1024, kPairTileVerts = 256;
struct PairPlan {
    int num_tiles = 0, num_pairs = 0;
    int64_t halo_slots = 0;
    std::vector<int32_t> tile_pair_ptr, tile_node_ptr, tile_nown, tile_nodes, tile_vert_ptr, tile_verts, tile_halo_off;
    // six words per pair: 14 node indices of 10 bits (three a word, the last two with the fifth
    // vertex index above them), four vertex indices of 8 bits.  Nodes: first cell's apex, the
    // face's vertices x, y, z, the apex's edges to them, edges xy, xz, yz, then the second cell's
    // apex and its edges to x, y, z; vertices: first apex, x, y, z, second apex.
    std::vector<uint32_t> records;
    std::vector<int32_t> cells;  // [num_pairs][2] mesh cells, -1: no second cell
    std::vector<int32_t> shared_node, shared_ptr, shared_slot;
};
// First cell's local basis -> pair slot is the identity; the second's (apex, x, z, y in its own
// orientation; edges (0,1), (0,2), (0,3), (1,2), (1,3), (2,3)):
constexpr int kPairSecond[10] = {10, 1, 3, 2, 11, 13, 12, 8, 7, 9};
// The slot indices of a record.
inline int pair_node(const uint32_t *w, int j) {
    return j < 12 ? (int)((w[j / 3] >> (10 * (j % 3))) & 1023u) : (int)((w[4] >> (10 * (j - 12))) & 1023u);
}
inline int pair_vert(const uint32_t *w, int j) { return j < 4 ? (int)((w[5] >> (8 * j)) & 255u) : (int)((w[4] >> 20) & 255u); }

// Pair plan of the base plan's cells (P2).  The cells are cut by recursive coordinate bisection of their
// centroids; where that gives no fewer halo slots than the base plan's tiles, those are kept.  Nonzero
// with a message where there is none (a tile of the base plan would need more than kPairTilePairs).
int build_pair_plan(const MeshView &m, const HostPlan &base, PairPlan *pp, std::string *err);

// Gather plan of a small key: tiles own nodes instead of cells.  Each tile holds every cell that touches
// one of its nodes (cells on tile boundaries appear in several tiles and are evaluated in each), so
// its sums are complete and nothing is left for a second pass: halo_slots = 0, and only the first
// tile_nown nodes of a tile's list are written.  `cells` repeats the duplicated cells.  At most
// max_tiles tiles of at most kGatherCells cells (one per thread); *fits is false, and the plan empty, when the key is too
// large for that.
constexpr int kGatherCells = 256;
int build_gather_plan(const MeshView &m, const HostPlan &base, int max_tiles, HostPlan *gp, bool *fits);

// sort_by_color: order each tile's cells by colour (colour-phase accumulation activates
// contiguous threads); otherwise cells keep their mesh order inside the tile (neighbouring
// threads then touch neighbouring nodes: structured LDS access for atomic accumulation).
// When the key's cells in input order tile badly (more than 1.5 halo slots per cell, e.g. a mesh
// numbered row by row), the cells are also tiled in Morton order of their centroids and the plan
// with fewer halo slots is kept.
// Permutation (new position -> point) listing n points [n][3] in Morton (Z-curve) order.
std::vector<int32_t> morton_permutation(const double *xyz, size_t n);

int build_host_plan(const MeshView &m, int label_value, const TileLimits &lim, HostPlan *hp,
                    std::string *err, bool sort_by_color = true);

}  // namespace plx
