// plx_plan.cpp -- tile plan of one weak-form key, built on the host (no device calls).
//
// The key's cells (PyLith's DSLabelAccess pointsIS: cells with the key's label value,
// feassemble/DSLabelAccess.icc:53-84) are cut, in cell order, into tiles bounded by the
// workgroup size and the LDS capacity.  Per tile: greedy cell colouring (cells sharing a node
// get different colours; cells sorted by colour), the node list with owned nodes first (numbered
// for LDS bank balance), 16-bit local closures, and halo slots for nodes other tiles also touch.
#include <algorithm>
#include <array>
#include <cmath>
#include <exception>
#include <iterator>
#include <mutex>
#include <numeric>
#include <system_error>
#include <thread>

#include "plx_plan.hpp"

namespace plx {

// Morton (Z-order) permutation of n points on a 2^21 grid over their bounding box (a finer grid
// than the mesh spacing, so points sharing a grid point are rare; ties keep input order).
std::vector<int32_t> morton_permutation(const double *xyz, size_t n) {
    double lo[3] = {1e300, 1e300, 1e300}, hi[3] = {-1e300, -1e300, -1e300};
    for (size_t i = 0; i < n; ++i)
        for (int d = 0; d < 3; ++d) {
            lo[d] = std::min(lo[d], xyz[3 * i + d]);
            hi[d] = std::max(hi[d], xyz[3 * i + d]);
        }
    const double span = std::max({hi[0] - lo[0], hi[1] - lo[1], hi[2] - lo[2], 1e-300});
    auto spread = [](uint64_t x) {  // 21 bits -> every third bit
        x &= 0x1fffff;
        x = (x | x << 32) & 0x1f00000000ffffull;
        x = (x | x << 16) & 0x1f0000ff0000ffull;
        x = (x | x << 8) & 0x100f00f00f00f00full;
        x = (x | x << 4) & 0x10c30c30c30c30c3ull;
        x = (x | x << 2) & 0x1249249249249249ull;
        return x;
    };
    std::vector<std::pair<uint64_t, int32_t>> key(n);
    for (size_t i = 0; i < n; ++i) {
        uint64_t code = 0;
        for (int d = 0; d < 3; ++d) {
            const double t = (xyz[3 * i + d] - lo[d]) / span;
            code |= spread((uint64_t)std::min(2097151.0, std::max(0.0, t * 2097151.0))) << d;
        }
        key[i] = {code, (int32_t)i};
    }
    std::stable_sort(key.begin(), key.end(),
                     [](const std::pair<uint64_t, int32_t> &a, const std::pair<uint64_t, int32_t> &b) {
                         return a.first < b.first;
                     });
    std::vector<int32_t> out(n);
    for (size_t i = 0; i < n; ++i) out[i] = key[i].second;
    return out;
}

// Joins its threads, whichever way the scope is left.
struct Threads {
    std::vector<std::thread> th;
    ~Threads() { join(); }
    void join() {
        for (auto &x : th)
            if (x.joinable()) x.join();
    }
};

// The first exception of work on several threads, to be thrown again by the one that started them.
struct FirstFailure {
    std::mutex mu;
    std::exception_ptr what;
    template <typename F>
    void guard(const F &work) {
        try {
            work();
        } catch (...) {
            std::lock_guard<std::mutex> lock(mu);
            if (!what) what = std::current_exception();
        }
    }
    void rethrow() const {
        if (what) std::rethrow_exception(what);
    }
};

// body(lo, hi) over [0, n) on host threads, in contiguous ranges.
template <typename F>
static void parallel_ranges(int n, const F &body) {
    const int nt = std::max(1, std::min({(int)std::thread::hardware_concurrency(), 16, n / 64 + 1}));
    FirstFailure failure;
    Threads threads;
    threads.th.reserve(nt);
    for (int t = 0; t < nt; ++t) {
        auto range = [&, t] {
            failure.guard([&] { body((int)((int64_t)n * t / nt), (int)((int64_t)n * (t + 1) / nt)); });
        };
        if (t + 1 == nt) {  // the last range runs here
            range();
            break;
        }
        try {
            threads.th.emplace_back(range);
        } catch (const std::system_error &) {  // no thread to be had: so does this one
            range();
        }
    }
    threads.join();
    failure.rethrow();
}

template <typename F>
static void parallel_for(int n, const F &body) {
    parallel_ranges(n, [&](int lo, int hi) {
        for (int i = lo; i < hi; ++i) body(i);
    });
}

// here() and there(), the latter on a thread of its own if `threaded` and one is to be had.
template <typename Here, typename There>
static void both(bool threaded, const Here &here, const There &there) {
    FirstFailure failure;
    Threads other;
    if (threaded) {
        other.th.reserve(1);
        try {
            other.th.emplace_back([&] { failure.guard(there); });
        } catch (const std::system_error &) {
            threaded = false;
        }
    }
    here();
    if (!threaded) there();
    other.join();
    failure.rethrow();
}

// v's distinct entries (non-negative), sorted.  Entries repeat several times over (a node in every cell around
// it): the repeats go first, through a table of twice the entries, and only the rest is sorted.
static int distinct(std::vector<int32_t> &v) {
    if (v.size() > 64) {
        int bits = 8;
        while (((size_t)1 << bits) < 2 * v.size()) ++bits;
        std::vector<int32_t> table((size_t)1 << bits, -1);
        size_t kept = 0;
        for (size_t i = 0; i < v.size(); ++i) {
            const int32_t x = v[i];
            size_t at = (uint32_t)x * 2654435769u >> (32 - bits);
            while (table[at] >= 0 && table[at] != x) at = (at + 1) & (table.size() - 1);
            if (table[at] == x) continue;
            table[at] = x;
            v[kept++] = x;
        }
        v.resize(kept);
    }
    std::sort(v.begin(), v.end());
    v.erase(std::unique(v.begin(), v.end()), v.end());
    return (int)v.size();
}

// Nodes that several tiles touch, ascending, and the ranges of their halo slots (empty: none).
static void shared_map(int num_nodes, const std::vector<int32_t> &tile_count, std::vector<int32_t> &node,
                       std::vector<int32_t> &ptr) {
    node.clear();
    ptr.assign(1, 0);
    for (int i = 0; i < num_nodes; ++i)
        if (tile_count[i] > 1) {
            node.push_back(i);
            ptr.push_back(ptr.back() + tile_count[i]);
        }
}

// The cells in Morton order of their centroids.
static std::vector<int32_t> morton_order(const MeshView &m, const std::vector<int32_t> &cells) {
    const size_t n = cells.size();
    std::vector<double> cen(3 * n);
    for (size_t i = 0; i < n; ++i) {
        const int32_t *cn = m.cone + (size_t)cells[i] * m.nv;
        for (int d = 0; d < 3; ++d) {
            double acc = 0.0;
            for (int v = 0; v < m.nv; ++v) acc += m.coords[3 * (size_t)cn[v] + d];
            cen[3 * i + d] = acc / m.nv;
        }
    }
    std::vector<int32_t> rank = morton_permutation(cen.data(), n), out(n);
    for (size_t i = 0; i < n; ++i) out[i] = cells[rank[i]];
    return out;
}

static int plan_cells(const MeshView &m, const TileLimits &lim, HostPlan *hp, std::string *err,
                      bool sort_by_color);

// LDS bank balance of a tile's local numbering.  The cell kernels address the staged arrays as
// [3 k + c] doubles, so an 8-byte access to local index k falls on bank pair (3 k + c) mod 16 of
// the 32 four-byte banks, which k mod 16 fixes.  A half-wave (32 consecutive cells of the tile)
// accesses slot b of its 32 cells in one instruction and takes as many cycles as its most loaded
// pair.  `ids` are the tile's items (nodes or vertices), `ranges` their position ranges (owned,
// then shared: an item keeps its range), and slot[b][i] the tile-local item of slot b of cell i.
// Items get residues mod 16 that spread every such access, greedily in order of decreasing use
// (each takes the residue its range still has room for that adds least to the summed squared
// loads of its accesses).  On return `ids` is reordered so that position p holds an item of
// residue p mod 16.
constexpr int kFixShared = 1;
static void balance_banks(std::vector<int32_t> &ids, const std::vector<int> &ranges,
                          const std::vector<std::vector<int32_t>> &slot, int ncell, int nfixed = 0) {
    const int n = (int)ids.size();
    if (n <= 16) return;
    // accesses: (half-wave, slot) -> its distinct items
    std::vector<int32_t> acc_ptr(1, 0), acc_items, item_acc_ptr(n + 1, 0), item_acc;
    std::vector<int32_t> seen(n, -1);
    int nacc = 0;
    for (int g = 0; g < ncell; g += 32)
        for (size_t b = 0; b < slot.size(); ++b, ++nacc) {
            for (int i = g; i < std::min(ncell, g + 32); ++i) {
                const int32_t k = slot[b][i];
                if (seen[k] != nacc) {
                    seen[k] = nacc;
                    acc_items.push_back(k);
                    item_acc_ptr[k + 1]++;
                }
            }
            acc_ptr.push_back((int32_t)acc_items.size());
        }
    for (int k = 0; k < n; ++k) item_acc_ptr[k + 1] += item_acc_ptr[k];
    item_acc.resize(acc_items.size());
    {
        std::vector<int32_t> fill(item_acc_ptr.begin(), item_acc_ptr.end() - 1);
        for (int a = 0; a < nacc; ++a)
            for (int j = acc_ptr[a]; j < acc_ptr[a + 1]; ++j) item_acc[fill[acc_items[j]]++] = a;
    }
    // residue capacities of each position range, the item's range
    const int nr = (int)ranges.size() - 1;
    std::vector<std::array<int, 16>> cap(nr);
    std::vector<int> range_of(n);
    for (int q = 0; q < nr; ++q) {
        cap[q].fill(0);
        for (int p = ranges[q]; p < ranges[q + 1]; ++p) {
            cap[q][p & 15]++;
            range_of[p] = q;
        }
    }
    std::vector<std::array<int16_t, 16>> load(nacc);
    for (auto &l : load) l.fill(0);
    std::vector<int> res(n, -1), order(n);
    for (int k = 0; k < n; ++k) order[k] = k;
    // the last nfixed ranges keep their positions (residue p mod 16)
    for (int k = 0; k < n; ++k)
        if (range_of[k] >= nr - nfixed) {
            res[k] = k & 15;
            cap[range_of[k]][k & 15]--;
            for (int j = item_acc_ptr[k]; j < item_acc_ptr[k + 1]; ++j) load[item_acc[j]][k & 15]++;
        }
    std::stable_sort(order.begin(), order.end(), [&](int a, int b) {
        return item_acc_ptr[a + 1] - item_acc_ptr[a] > item_acc_ptr[b + 1] - item_acc_ptr[b];
    });
    for (int k : order) {
        if (res[k] >= 0) continue;
        const int q = range_of[k];
        int sum[16] = {};
        for (int j = item_acc_ptr[k]; j < item_acc_ptr[k + 1]; ++j)
            for (int r = 0; r < 16; ++r) sum[r] += load[item_acc[j]][r];
        int best = -1;
        for (int r = 0; r < 16; ++r)
            if (cap[q][r] > 0 && (best < 0 || sum[r] < sum[best])) best = r;
        res[k] = best;
        cap[q][best]--;
        for (int j = item_acc_ptr[k]; j < item_acc_ptr[k + 1]; ++j) load[item_acc[j]][best]++;
    }
    // positions: within each range, residue r takes positions p = r (mod 16)
    std::vector<int32_t> out(n);
    for (int q = 0; q < nr; ++q) {
        std::array<std::vector<int>, 16> byres;
        for (int k = 0; k < n; ++k)
            if (range_of[k] == q) byres[res[k]].push_back(k);
        std::array<size_t, 16> next{};
        for (int p = ranges[q]; p < ranges[q + 1]; ++p) out[p] = ids[byres[p & 15][next[p & 15]++]];
    }
    ids.swap(out);
}

int build_host_plan(const MeshView &m, int label_value, const TileLimits &lim, HostPlan *hp,
                    std::string *err, bool sort_by_color) {
    std::vector<int32_t> &cells = hp->cells;
    cells.clear();
    for (int c = 0; c < m.num_cells; ++c)
        if ((m.labels ? m.labels[c] : 0) == label_value) cells.push_back(c);
    if (cells.empty()) {
        *err = "no cells carry the key's label value";
        return 1;
    }
    const std::vector<int32_t> input = cells;
    int e = plan_cells(m, lim, hp, err, sort_by_color);
    hp->reordered = false;
    if (e || !m.coords || (double)hp->halo_slots <= 1.5 * (double)input.size()) return e;
    HostPlan alt;
    alt.cells = morton_order(m, input);
    std::string err2;
    if (plan_cells(m, lim, &alt, &err2, sort_by_color) == 0 && alt.halo_slots < hp->halo_slots) {
        *hp = std::move(alt);
        hp->reordered = true;
    }
    return 0;
}

// The plan of hp->cells taken in their given order.
static int plan_cells(const MeshView &m, const TileLimits &lim, HostPlan *hp, std::string *err,
                      bool sort_by_color) {
    const int nb = m.nb, nv = m.nv;
    std::vector<int32_t> &cells = hp->cells;
    const int ncells = (int)cells.size();

    // Greedy tiling in cell order, bounded by LDS capacity.
    std::vector<int32_t> node_mark(m.num_nodes, -1), vert_mark(m.num_vertices, -1);
    std::vector<int32_t> &tile_cell_ptr = hp->tile_cell_ptr;
    tile_cell_ptr.assign(1, 0);
    {
        int tcells = 0, tnodes = 0, tverts = 0, tile = 0;
        for (int i = 0; i < ncells; ++i) {
            const int32_t *cl = m.closure + (size_t)cells[i] * nb;
            const int32_t *cn = m.cone + (size_t)cells[i] * nv;
            int newn = 0, newv = 0;
            for (int b = 0; b < nb; ++b) newn += node_mark[cl[b]] != tile;
            for (int b = 0; b < nv; ++b) newv += vert_mark[cn[b]] != tile;
            if (tcells == lim.cells || tnodes + newn > lim.nodes || tverts + newv > lim.verts) {
                tile_cell_ptr.push_back(i);
                tcells = tnodes = tverts = 0;
                ++tile;
            }
            for (int b = 0; b < nb; ++b)
                if (node_mark[cl[b]] != tile) {
                    node_mark[cl[b]] = tile;
                    ++tnodes;
                }
            for (int b = 0; b < nv; ++b)
                if (vert_mark[cn[b]] != tile) {
                    vert_mark[cn[b]] = tile;
                    ++tverts;
                }
            ++tcells;
        }
        tile_cell_ptr.push_back(ncells);
    }
    const int ntiles = (int)tile_cell_ptr.size() - 1;
    hp->num_tiles = ntiles;

    // Each tile by itself, on host threads: its sorted nodes, colouring, node and vertex lists, local
    // closures; then the tiles one after another.
    struct Tile {
        std::vector<int32_t> nodes, own, ids, verts;  // sorted nodes; owned ones; local order (owned, shared); vertices
        int ncolor = 0;
    };
    std::vector<Tile> tiles(ntiles);
    parallel_for(ntiles, [&](int t) {
        std::vector<int32_t> &v = tiles[t].nodes;
        for (int i = tile_cell_ptr[t]; i < tile_cell_ptr[t + 1]; ++i)
            v.insert(v.end(), m.closure + (size_t)cells[i] * nb, m.closure + (size_t)(cells[i] + 1) * nb);
        distinct(v);
    });
    std::vector<int32_t> tile_count(m.num_nodes, 0);  // how many tiles touch each node
    for (const Tile &T : tiles)
        for (int32_t x : T.nodes) ++tile_count[x];
    hp->color.assign(ncells, 0);
    hp->lclosure.assign((size_t)nb * ncells, 0);
    hp->lcone.assign((size_t)nv * ncells, 0);
    std::vector<char> too_many(ntiles, 0);
    parallel_for(ntiles, [&](int t) {
        Tile &T = tiles[t];
        const int c0 = tile_cell_ptr[t], tc = tile_cell_ptr[t + 1] - c0;
        auto local = [](const std::vector<int32_t> &v, int32_t x) {
            return (int32_t)(std::lower_bound(v.begin(), v.end(), x) - v.begin());
        };
        // greedy colouring, then cells sorted by colour
        std::vector<int32_t> lc((size_t)tc * nb);  // sorted position of each closure node
        for (int i = 0; i < tc; ++i)
            for (int b = 0; b < nb; ++b) lc[(size_t)i * nb + b] = local(T.nodes, m.closure[(size_t)cells[c0 + i] * nb + b]);
        std::vector<std::array<uint64_t, 2>> used(T.nodes.size(), {0, 0});
        std::vector<std::pair<int, int32_t>> order;  // colour, cell of the tile
        for (int i = 0; i < tc; ++i) {
            uint64_t m0 = 0, m1 = 0;
            for (int b = 0; b < nb; ++b) {
                m0 |= used[lc[(size_t)i * nb + b]][0];
                m1 |= used[lc[(size_t)i * nb + b]][1];
            }
            int c = 0;
            while (c < 128 && ((c < 64 ? (m0 >> c) : (m1 >> (c - 64))) & 1)) ++c;
            if (c >= 128) {
                too_many[t] = 1;
                return;
            }
            for (int b = 0; b < nb; ++b) used[lc[(size_t)i * nb + b]][c >> 6] |= (uint64_t)1 << (c & 63);
            order.emplace_back(c, i);
            T.ncolor = std::max(T.ncolor, c + 1);
        }
        if (sort_by_color)
            std::stable_sort(order.begin(), order.end(),
                             [](const std::pair<int, int32_t> &a, const std::pair<int, int32_t> &b) {
                                 return a.first < b.first;
                             });
        {
            std::vector<int32_t> sorted(tc), lsorted(lc.size());
            for (int i = 0; i < tc; ++i) {
                hp->color[c0 + i] = (uint8_t)order[i].first;
                sorted[i] = cells[c0 + order[i].second];
                std::copy_n(&lc[(size_t)order[i].second * nb], nb, &lsorted[(size_t)i * nb]);
            }
            std::copy(sorted.begin(), sorted.end(), cells.begin() + c0);
            lc.swap(lsorted);
        }
        // local numbering: owned nodes, then shared ones.  Colour-sorted tiles put scattered cells in
        // each half-wave: their owned nodes are numbered for LDS bank balance around the shared
        // ones, which keep node order (the halo reduction reads their partials in node order).
        // Tiles in mesh order keep node order: neighbouring lanes already touch spread-out banks.
        std::vector<int32_t> sh;
        for (int32_t x : T.nodes) (tile_count[x] == 1 ? T.own : sh).push_back(x);
        T.ids = T.own;
        T.ids.insert(T.ids.end(), sh.begin(), sh.end());
        std::vector<int32_t> rank(T.ids.size());  // sorted position -> local index
        auto ranks = [&] {
            for (size_t k = 0; k < T.ids.size(); ++k) rank[local(T.nodes, T.ids[k])] = (int32_t)k;
        };
        ranks();
        if (sort_by_color) {
            std::vector<std::vector<int32_t>> slot(nb, std::vector<int32_t>(tc));
            for (int i = 0; i < tc; ++i)
                for (int b = 0; b < nb; ++b) slot[b][i] = rank[lc[(size_t)i * nb + b]];
            balance_banks(T.ids, {0, (int)T.own.size(), (int)T.ids.size()}, slot, tc, kFixShared);
            ranks();
        }
        for (int i = 0; i < tc; ++i)
            for (int b = 0; b < nb; ++b) hp->lclosure[(size_t)b * ncells + c0 + i] = (uint16_t)rank[lc[(size_t)i * nb + b]];
        if (m.cone_is_closure) return;
        std::vector<int32_t> vs;
        for (int i = 0; i < tc; ++i)
            vs.insert(vs.end(), m.cone + (size_t)cells[c0 + i] * nv, m.cone + (size_t)(cells[c0 + i] + 1) * nv);
        distinct(vs);
        T.verts = vs;
        std::vector<std::vector<int32_t>> slot(nv, std::vector<int32_t>(tc));
        for (int i = 0; i < tc; ++i)
            for (int b = 0; b < nv; ++b) slot[b][i] = local(vs, m.cone[(size_t)cells[c0 + i] * nv + b]);
        if (sort_by_color && vs.size() > 16) balance_banks(T.verts, {0, (int)vs.size()}, slot, tc);
        std::vector<int32_t> vrank(vs.size());
        for (size_t k = 0; k < vs.size(); ++k) vrank[local(vs, T.verts[k])] = (int32_t)k;
        for (int i = 0; i < tc; ++i)
            for (int b = 0; b < nv; ++b) hp->lcone[(size_t)b * ncells + c0 + i] = (uint16_t)vrank[slot[b][i]];
    });
    hp->tile_ncolor.clear();
    hp->max_colors = 0;
    hp->tile_node_ptr.assign(1, 0);
    hp->tile_vert_ptr.assign(1, 0);
    hp->tile_nown.clear();
    hp->tile_nodes.clear();
    hp->tile_verts.clear();
    hp->tile_halo_off.clear();
    int64_t halo = 0;
    int max_nodes = 0, max_verts = 0;
    for (int t = 0; t < ntiles; ++t) {
        if (too_many[t]) {
            *err = "tile colouring needs more than 128 colours";
            return 1;
        }
        const Tile &T = tiles[t];
        hp->tile_ncolor.push_back(T.ncolor);
        hp->max_colors = std::max(hp->max_colors, T.ncolor);
        hp->tile_nown.push_back((int32_t)T.own.size());
        hp->tile_halo_off.push_back((int32_t)halo);
        halo += (int64_t)(T.ids.size() - T.own.size());
        hp->tile_nodes.insert(hp->tile_nodes.end(), T.ids.begin(), T.ids.end());
        hp->tile_verts.insert(hp->tile_verts.end(), T.verts.begin(), T.verts.end());
        hp->tile_node_ptr.push_back((int32_t)hp->tile_nodes.size());
        hp->tile_vert_ptr.push_back((int32_t)hp->tile_verts.size());
        max_nodes = std::max(max_nodes, (int)T.ids.size());
        max_verts = std::max(max_verts, (int)T.verts.size());
    }
    if (m.cone_is_closure) {
        hp->tile_verts = hp->tile_nodes;
        hp->tile_vert_ptr = hp->tile_node_ptr;
        hp->lcone = hp->lclosure;
        max_verts = max_nodes;
    }
    if (halo > INT32_MAX) {
        *err = "halo too large";
        return 1;
    }
    hp->halo_slots = halo;
    hp->max_nodes = max_nodes;
    hp->max_verts = max_verts;

    // Shared-node reduction map: nodes ascending, slots in tile order.
    shared_map(m.num_nodes, tile_count, hp->shared_node, hp->shared_ptr);
    std::vector<int32_t> place(m.num_nodes, -1);
    for (size_t i = 0; i < hp->shared_node.size(); ++i) place[hp->shared_node[i]] = hp->shared_ptr[i];
    hp->shared_slot.resize((size_t)halo);
    int32_t slot = 0;
    for (const Tile &T : tiles)
        for (size_t k = T.own.size(); k < T.ids.size(); ++k) hp->shared_slot[place[T.ids[k]]++] = slot++;
    return 0;
}

// --------------------------------------------------------------------------------------------
// Pair plan.
// --------------------------------------------------------------------------------------------

namespace {
struct PairTile {
    int n = 0;                              // cells
    std::vector<std::array<int, 4>> match;  // pairs: first cell, second (-1: none), their vertices opposite the face
    int npaired = 0;                        // those with a second cell come first
    std::vector<int32_t> nodes;  // sorted distinct, then in local order (owned, shared)
    std::vector<int32_t> verts;  // likewise
    std::vector<std::array<int, 4>> cv;  // each cell's vertices, places in the sorted verts
    int nown = 0;
    std::vector<int32_t> cells;  // [pairs][2]
    std::vector<uint32_t> rec;
};
}  // namespace

// Position of x in the sorted v.
static int place_of(const std::vector<int32_t> &v, int32_t x) {
    return (int)(std::lower_bound(v.begin(), v.end(), x) - v.begin());
}

// Local node of the edge between two vertices of a P2 tetrahedron.
static const int kTetEdge[4][4] = {{-1, 4, 5, 6}, {4, -1, 7, 8}, {5, 7, -1, 9}, {6, 8, 9, -1}};

// Local vertices of cells a and b, which share a face, the vertices opposite it (oa, ob) first and b's
// face turned so that its first vertex is a's; the other two then run the opposite way round in a
// consistently oriented mesh.  False, and the cells no pair, where they do not, or where the cells'
// nodes on the face differ (vertices of one place with nodes of their own on either side).
static bool turn_to_face(const MeshView &m, int32_t a, int oa, int32_t b, int ob, int pa[4], int pb[4]) {
    static const int kApex[4][4] = {{0, 1, 2, 3}, {1, 0, 3, 2}, {2, 0, 1, 3}, {3, 0, 2, 1}};  // even permutations
    const int32_t *va = m.cone + 4 * (size_t)a, *vb = m.cone + 4 * (size_t)b;
    const int32_t *ca = m.closure + 10 * (size_t)a, *cb = m.closure + 10 * (size_t)b;
    for (int k = 0; k < 4; ++k) pa[k] = kApex[oa][k];
    for (int r = 0; r < 3; ++r) {
        pb[0] = kApex[ob][0];
        for (int k = 0; k < 3; ++k) pb[1 + k] = kApex[ob][1 + (k + r) % 3];
        if (vb[pb[1]] == va[pa[1]]) break;
    }
    const int qb[4] = {pb[0], pb[1], pb[3], pb[2]};  // b's vertices in a's order
    for (int k = 1; k < 4; ++k) {
        if (vb[qb[k]] != va[pa[k]] || cb[qb[k]] != ca[pa[k]]) return false;
        const int l = k % 3 + 1;  // and the edge to the next
        if (cb[kTetEdge[qb[k]][qb[l]]] != ca[kTetEdge[pa[k]][pa[l]]]) return false;
    }
    return true;
}

// The vertices (unless there) and pairs of the cells ids[0 .. n).
static void match_cells(const MeshView &m, const int32_t *ids, int n, PairTile &T) {
    T.n = n;
    if (T.verts.empty())
        for (int i = 0; i < n; ++i) T.verts.insert(T.verts.end(), m.cone + 4 * (size_t)ids[i], m.cone + 4 * (size_t)(ids[i] + 1));
    distinct(T.verts);
    T.cv.resize(n);
    // faces of the tile: (vertices sorted) -> cell and the vertex opposite
    std::vector<std::pair<uint64_t, int32_t>> faces;
    faces.reserve(4 * (size_t)n);
    for (int i = 0; i < n; ++i) {
        std::array<int, 4> &v = T.cv[i];
        for (int k = 0; k < 4; ++k) v[k] = place_of(T.verts, m.cone[4 * (size_t)ids[i] + k]);
        for (int k = 0; k < 4; ++k) {
            std::array<int, 3> f{v[(k + 1) & 3], v[(k + 2) & 3], v[(k + 3) & 3]};
            std::sort(f.begin(), f.end());
            faces.push_back({((uint64_t)f[0] << 40) | ((uint64_t)f[1] << 20) | (uint64_t)f[2], 4 * i + k});
        }
    }
    std::sort(faces.begin(), faces.end());
    std::vector<std::array<std::array<int, 3>, 4>> nbr(n);  // (neighbour, my opposite vertex, its)
    std::vector<int> deg(n, 0);
    for (size_t f = 0; f + 1 < faces.size(); ++f)
        if (faces[f].first == faces[f + 1].first) {
            const int a = faces[f].second >> 2, b = faces[f + 1].second >> 2;
            if (a != b && deg[a] < 4 && deg[b] < 4) {
                nbr[a][deg[a]++] = {b, faces[f].second & 3, faces[f + 1].second & 3};
                nbr[b][deg[b]++] = {a, faces[f + 1].second & 3, faces[f].second & 3};
            }
            ++f;
        }
    // matching: cells with the fewest free neighbours first, each to its neighbour with the fewest
    std::vector<int> mate(n, -1), free_deg(deg);
    std::array<std::vector<int>, 5> bucket;
    for (int i = n - 1; i >= 0; --i) bucket[free_deg[i]].push_back(i);
    T.match.clear();
    for (int d = 1; d <= 4;) {
        if (bucket[d].empty()) {
            ++d;
            continue;
        }
        const int a = bucket[d].back();
        bucket[d].pop_back();
        if (mate[a] >= 0 || free_deg[a] != d) continue;
        int best = -1;
        for (int k = 0; k < deg[a]; ++k) {
            const int b = nbr[a][k][0];
            if (mate[b] >= 0) continue;
            int pa[4], pb[4];
            if (!turn_to_face(m, ids[a], nbr[a][k][1], ids[b], nbr[a][k][2], pa, pb)) continue;
            if (best < 0 || free_deg[b] < free_deg[nbr[a][best][0]]) best = k;
        }
        if (best < 0) continue;  // no neighbour it can be turned to: stays single
        const int b = nbr[a][best][0];
        mate[a] = b;
        mate[b] = a;
        T.match.push_back({a, b, nbr[a][best][1], nbr[a][best][2]});
        for (int c : {a, b})
            for (int k = 0; k < deg[c]; ++k) {
                const int e = nbr[c][k][0];
                if (mate[e] >= 0) continue;
                if (--free_deg[e] > 0) bucket[free_deg[e]].push_back(e);
                if (free_deg[e] > 0 && free_deg[e] < d) d = free_deg[e];
            }
    }
    T.npaired = (int)T.match.size();
    for (int i = 0; i < n; ++i)
        if (mate[i] < 0) T.match.push_back({i, -1, 0, 0});
}

// Cells order[0 .. n) cut into tiles by recursive bisection of their centroids along the longest
// axis; the tiles, their cells paired, are appended to `tiles` in order.  A cell left alone takes a
// pair's place: a part of up to 2 kPairTilePairs cells that does not fit with its pairs is cut on.  A cut
// may move by a sixteenth of its range to the widest gap between centroids there: between layers of
// cells where the mesh has them.
static void bisect(const MeshView &m, const std::vector<double> &cen, int32_t *order, int n, std::vector<PairTile> &tiles_out,
                   int depth) {
    const int most = 2 * kPairTilePairs;
    if (n <= most) {
        std::vector<int32_t> nodes, verts;
        nodes.reserve((size_t)n * m.nb);
        verts.reserve((size_t)n * m.nv);
        for (int i = 0; i < n; ++i) {
            const int32_t c = order[i];
            nodes.insert(nodes.end(), m.closure + (size_t)c * m.nb, m.closure + (size_t)(c + 1) * m.nb);
            verts.insert(verts.end(), m.cone + (size_t)c * m.nv, m.cone + (size_t)(c + 1) * m.nv);
        }
        distinct(nodes);
        distinct(verts);
        if (n == 1 || ((int)nodes.size() <= kPairTileNodes && (int)verts.size() <= kPairTileVerts)) {
            PairTile T;
            T.nodes = std::move(nodes);
            T.verts = std::move(verts);
            match_cells(m, order, n, T);
            if ((int)T.match.size() <= kPairTilePairs) {
                tiles_out.push_back(std::move(T));
                return;
            }
        }
    }
    double lo[3] = {1e300, 1e300, 1e300}, hi[3] = {-1e300, -1e300, -1e300};
    for (int i = 0; i < n; ++i)
        for (int d = 0; d < 3; ++d) {
            lo[d] = std::min(lo[d], cen[3 * (size_t)order[i] + d]);
            hi[d] = std::max(hi[d], cen[3 * (size_t)order[i] + d]);
        }
    int ax = 0;
    for (int d = 1; d < 3; ++d)
        if (hi[d] - lo[d] > hi[ax] - lo[ax]) ax = d;
    auto less = [&](int32_t a, int32_t b) {
        const double x = cen[3 * (size_t)a + ax], y = cen[3 * (size_t)b + ax];
        return x < y || (x == y && a < b);
    };
    // two parts holding whole numbers of nearly full tiles (15 / 16 of the bound)
    const int tiles = std::max(2, (n + most * 15 / 16 - 1) / (most * 15 / 16));
    const int ideal = std::min(n - 1, std::max(1, (int)((int64_t)n * (tiles / 2) / tiles)));
    const int w = n / 16;
    const int a = std::max(1, ideal - w), b = std::min(n - 1, ideal + w);
    std::nth_element(order, order + a, order + n, less);
    if (b > a) std::nth_element(order + a, order + b, order + n, less);
    std::sort(order + a, order + b, less);
    int cut = ideal;
    double widest = 0.0;
    for (int i = a; i <= b; ++i) {
        if (i > a && i >= b && b == a) break;
        const double below = i == a ? -1e300 : cen[3 * (size_t)order[i - 1] + ax];
        const double gap = i == a ? 0.0 : cen[3 * (size_t)order[i] + ax] - below;
        if (gap > 1.001 * widest || (gap > 0.999 * widest && std::abs(i - ideal) < std::abs(cut - ideal) && gap > 0.0)) {
            widest = std::max(widest, gap);
            cut = i;
        }
    }
    std::vector<PairTile> right;
    both(depth < 3, [&] { bisect(m, cen, order, cut, tiles_out, depth + 1); },
         [&] { bisect(m, cen, order + cut, n - cut, right, depth + 1); });
    std::move(right.begin(), right.end(), std::back_inserter(tiles_out));
}

// Numbering and records of one tile (cells ids[0 .. T.n), paired; T.nodes its sorted nodes).
static void build_pair_tile(const MeshView &m, const int32_t *ids, const std::vector<int32_t> &tile_count, PairTile &T) {
    const int np = (int)T.match.size();
    const std::vector<int32_t> verts(std::move(T.verts));
    const std::vector<std::array<int, 4>> cv(std::move(T.cv));
    // slots: mesh nodes [14] and tile vertices [5] of each pair
    std::vector<std::array<int32_t, 14>> pn(np);
    std::vector<std::array<int, 5>> pv(np);
    for (int p = 0; p < np; ++p) {
        const int a = T.match[p][0], b = T.match[p][1];
        int pa[4] = {0, 1, 2, 3}, pb[4] = {0, 1, 3, 2};
        if (b >= 0) (void)turn_to_face(m, ids[a], T.match[p][2], ids[b], T.match[p][3], pa, pb);
        const int q = b >= 0 ? b : a;  // alone: the second cell is the mirror image of the first
        const int32_t *ca = m.closure + 10 * (size_t)ids[a], *cb = m.closure + 10 * (size_t)ids[q];
        for (int k = 0; k < 4; ++k) {
            pn[p][k] = ca[pa[k]];
            pv[p][k] = cv[a][pa[k]];
        }
        for (int k = 0; k < 3; ++k) pn[p][4 + k] = ca[kTetEdge[pa[0]][pa[1 + k]]];
        pn[p][7] = ca[kTetEdge[pa[1]][pa[2]]];
        pn[p][8] = ca[kTetEdge[pa[1]][pa[3]]];
        pn[p][9] = ca[kTetEdge[pa[2]][pa[3]]];
        pn[p][10] = cb[pb[0]];
        pv[p][4] = cv[q][pb[0]];
        pn[p][11] = cb[kTetEdge[pb[0]][pb[1]]];  // to x
        pn[p][12] = cb[kTetEdge[pb[0]][pb[3]]];  // to y
        pn[p][13] = cb[kTetEdge[pb[0]][pb[2]]];  // to z
    }
    // pairs of one colour share no node; sorted by colour (paired ones first) a wave's atomic
    // targets are distinct
    std::vector<std::array<int32_t, 14>> pl(np);
    for (int p = 0; p < np; ++p)
        for (int j = 0; j < 14; ++j) pl[p][j] = place_of(T.nodes, pn[p][j]);
    std::vector<int> color(np), order(np);
    {
        std::vector<std::array<uint64_t, 2>> used(T.nodes.size(), {0, 0});
        for (int p = 0; p < np; ++p) {
            uint64_t m0 = 0, m1 = 0;
            for (int32_t k : pl[p]) {
                m0 |= used[k][0];
                m1 |= used[k][1];
            }
            int c = 0;
            while (c < 127 && ((c < 64 ? (m0 >> c) : (m1 >> (c - 64))) & 1)) ++c;
            for (int32_t k : pl[p]) used[k][c >> 6] |= (uint64_t)1 << (c & 63);
            color[p] = c + (p < T.npaired ? 0 : 128);
            order[p] = p;
        }
        std::stable_sort(order.begin(), order.end(), [&](int a, int b) { return color[a] < color[b]; });
    }
    // local numbering: owned nodes balanced over the LDS banks around the shared ones, which keep node
    // order (the halo reduction reads their partials in that order); vertices balanced
    std::vector<int32_t> own, sh, ord;
    for (int32_t x : T.nodes) (tile_count[x] == 1 ? own : sh).push_back(x);
    T.nown = (int)own.size();
    ord = own;
    ord.insert(ord.end(), sh.begin(), sh.end());
    std::vector<int32_t> rank(T.nodes.size());  // sorted position -> local index
    auto ranks = [&](const std::vector<int32_t> &v) {
        for (size_t k = 0; k < v.size(); ++k) rank[place_of(T.nodes, v[k])] = (int32_t)k;
    };
    ranks(ord);
    std::vector<std::vector<int32_t>> slot(14, std::vector<int32_t>(np));
    for (int i = 0; i < np; ++i)
        for (int j = 0; j < 14; ++j) slot[j][i] = rank[pl[order[i]][j]];
    balance_banks(ord, {0, T.nown, (int)ord.size()}, slot, np, kFixShared);
    ranks(ord);
    std::vector<int32_t> vo(verts.size()), vslot_id(verts.size());
    for (size_t k = 0; k < verts.size(); ++k) vo[k] = (int32_t)k;
    std::vector<std::vector<int32_t>> vslot(5, std::vector<int32_t>(np));
    for (int i = 0; i < np; ++i)
        for (int j = 0; j < 5; ++j) vslot[j][i] = pv[order[i]][j];
    balance_banks(vo, {0, (int)vo.size()}, vslot, np);
    for (size_t k = 0; k < vo.size(); ++k) vslot_id[vo[k]] = (int32_t)k;
    T.verts.resize(verts.size());
    for (size_t k = 0; k < vo.size(); ++k) T.verts[k] = verts[vo[k]];
    T.rec.assign(6 * (size_t)np, 0);
    T.cells.resize(2 * (size_t)np);
    for (int i = 0; i < np; ++i) {
        const int p = order[i];
        uint32_t *w = &T.rec[6 * (size_t)i];
        for (int j = 0; j < 12; ++j) w[j / 3] |= (uint32_t)rank[pl[p][j]] << (10 * (j % 3));
        w[4] = (uint32_t)rank[pl[p][12]] | (uint32_t)rank[pl[p][13]] << 10 | (uint32_t)vslot_id[pv[p][4]] << 20;
        for (int j = 0; j < 4; ++j) w[5] |= (uint32_t)vslot_id[pv[p][j]] << (8 * j);
        T.cells[2 * (size_t)i] = ids[T.match[p][0]];
        T.cells[2 * (size_t)i + 1] = T.match[p][1] >= 0 ? ids[T.match[p][1]] : -1;
    }
    T.nodes = std::move(ord);
}

// Halo slots of cells cut into the given tiles; per tile its sorted nodes, per node its tiles.
static int64_t tile_nodes_of(const MeshView &m, const std::vector<int32_t> &cells, const std::vector<int32_t> &ptr,
                             std::vector<PairTile> &tiles, std::vector<int32_t> &tile_count) {
    const int nt = (int)ptr.size() - 1;
    parallel_for(nt, [&](int t) {
        std::vector<int32_t> &v = tiles[t].nodes;
        if (!v.empty()) return;
        for (int i = ptr[t]; i < ptr[t + 1]; ++i)
            v.insert(v.end(), m.closure + (size_t)cells[i] * m.nb, m.closure + (size_t)(cells[i] + 1) * m.nb);
        distinct(v);
    });
    tile_count.assign(m.num_nodes, 0);
    for (const PairTile &T : tiles)
        for (int32_t x : T.nodes) ++tile_count[x];
    int64_t halo = 0;
    for (int32_t c : tile_count) halo += c > 1 ? c : 0;
    return halo;
}

int build_pair_plan(const MeshView &m, const HostPlan &base, PairPlan *pp, std::string *err) {
    if (m.nb != 10 || m.nv != 4 || !m.coords) {
        *err = "pair plans are for P2 tetrahedra";
        return 1;
    }
    const int n = (int)base.cells.size();
    std::vector<int32_t> cells(base.cells), ptr(1, 0);
    std::vector<PairTile> tiles;
    std::vector<int32_t> tile_count;
    {
        std::vector<double> cen(3 * (size_t)m.num_cells);
        for (int32_t c : cells)
            for (int d = 0; d < 3; ++d) {
                double acc = 0.0;
                for (int v = 0; v < 4; ++v) acc += m.coords[3 * (size_t)m.cone[4 * (size_t)c + v] + d];
                cen[3 * (size_t)c + d] = 0.25 * acc;
            }
        bisect(m, cen, cells.data(), n, tiles, 0);
        for (const PairTile &T : tiles) ptr.push_back(ptr.back() + T.n);
    }
    int64_t halo = tile_nodes_of(m, cells, ptr, tiles, tile_count);
    if (halo > base.halo_slots) {
        cells = base.cells;
        ptr = base.tile_cell_ptr;
        tiles.assign(base.num_tiles, PairTile());
        parallel_for(base.num_tiles, [&](int t) { match_cells(m, &cells[ptr[t]], ptr[t + 1] - ptr[t], tiles[t]); });
        for (const PairTile &T : tiles)
            if ((int)T.match.size() > kPairTilePairs) {
                *err = "pair tile over its bounds";
                return 1;
            }
        halo = tile_nodes_of(m, cells, ptr, tiles, tile_count);
    }
    const int nt = (int)ptr.size() - 1;
    parallel_for(nt, [&](int t) { build_pair_tile(m, &cells[ptr[t]], tile_count, tiles[t]); });
    *pp = PairPlan();
    pp->num_tiles = nt;
    pp->halo_slots = halo;
    pp->tile_pair_ptr.assign(1, 0);
    pp->tile_node_ptr.assign(1, 0);
    pp->tile_vert_ptr.assign(1, 0);
    // shared nodes ascending, their slots in tile order
    shared_map(m.num_nodes, tile_count, pp->shared_node, pp->shared_ptr);
    std::vector<int32_t> place(m.num_nodes, -1);
    for (size_t i = 0; i < pp->shared_node.size(); ++i) place[pp->shared_node[i]] = pp->shared_ptr[i];
    pp->shared_slot.resize((size_t)halo);
    int64_t off = 0;
    for (PairTile &T : tiles) {
        if ((int)T.nodes.size() > kPairTileNodes || (int)T.verts.size() > kPairTileVerts ||
            (int)T.cells.size() > 2 * kPairTilePairs || off > INT32_MAX) {
            *err = "pair tile over its bounds";
            return 1;
        }
        pp->tile_nown.push_back(T.nown);
        pp->tile_halo_off.push_back((int32_t)off);
        for (size_t k = (size_t)T.nown; k < T.nodes.size(); ++k) pp->shared_slot[place[T.nodes[k]]++] = (int32_t)off++;
        pp->tile_nodes.insert(pp->tile_nodes.end(), T.nodes.begin(), T.nodes.end());
        pp->tile_verts.insert(pp->tile_verts.end(), T.verts.begin(), T.verts.end());
        pp->cells.insert(pp->cells.end(), T.cells.begin(), T.cells.end());
        pp->records.insert(pp->records.end(), T.rec.begin(), T.rec.end());
        pp->tile_pair_ptr.push_back((int32_t)(pp->cells.size() / 2));
        pp->tile_node_ptr.push_back((int32_t)pp->tile_nodes.size());
        pp->tile_vert_ptr.push_back((int32_t)pp->tile_verts.size());
    }
    pp->num_pairs = (int)(pp->cells.size() / 2);
    return 0;
}

// --------------------------------------------------------------------------------------------
// Gather plan.
// --------------------------------------------------------------------------------------------

// order[0 .. n) cut into `parts` equal parts by bisection along the longest axis; sizes appended in order.
static void bisect_equal(const std::vector<double> &x, int32_t *order, int n, int parts, std::vector<int32_t> &sizes,
                         int depth = 0) {
    if (parts <= 1 || n <= 1) {
        sizes.push_back(n);
        return;
    }
    double lo[3] = {1e300, 1e300, 1e300}, hi[3] = {-1e300, -1e300, -1e300};
    for (int i = 0; i < n; ++i)
        for (int d = 0; d < 3; ++d) {
            lo[d] = std::min(lo[d], x[3 * (size_t)order[i] + d]);
            hi[d] = std::max(hi[d], x[3 * (size_t)order[i] + d]);
        }
    int ax = 0;
    for (int d = 1; d < 3; ++d)
        if (hi[d] - lo[d] > hi[ax] - lo[ax]) ax = d;
    const int left = parts / 2;
    const int cut = std::max(1, (int)((int64_t)n * left / parts));
    std::nth_element(order, order + cut, order + n, [&](int32_t a, int32_t b) {
        const double u = x[3 * (size_t)a + ax], v = x[3 * (size_t)b + ax];
        return u < v || (u == v && a < b);
    });
    std::vector<int32_t> right;
    both(depth < 3 && n > 2000, [&] { bisect_equal(x, order, cut, left, sizes, depth + 1); },
         [&] { bisect_equal(x, order + cut, n - cut, parts - left, right, depth + 1); });
    sizes.insert(sizes.end(), right.begin(), right.end());
}

int build_gather_plan(const MeshView &m, const HostPlan &base, int max_tiles, HostPlan *gp, bool *fits) {
    *fits = false;
    *gp = HostPlan();
    const int nb = m.nb, nv = m.nv;
    // (an early way out: boxes of up to 38^3 hexes or 6 x 16^3 tets fit 512 tiles)
    if (!m.coords || (int64_t)base.cells.size() > (int64_t)max_tiles * (nb == 8 ? 128 : 64)) return 0;
    // the key's cells and nodes, ascending; by their places there: each cell's nodes, each node's position (mean
    // of the incident cells' centroids) and incident cells
    std::vector<int32_t> cells(base.cells), nodes, rank(m.num_nodes, -1);
    std::sort(cells.begin(), cells.end());
    const int ncell = (int)cells.size();
    for (int32_t c : cells)
        for (int b = 0; b < nb; ++b) rank[m.closure[(size_t)c * nb + b]] = 0;
    for (int i = 0; i < m.num_nodes; ++i)
        if (rank[i] == 0) {
            rank[i] = (int32_t)nodes.size();
            nodes.push_back(i);
        }
    const int nnode = (int)nodes.size();
    std::vector<int32_t> cl((size_t)ncell * nb), ptr(nnode + 1, 0), inc;
    std::vector<double> x(3 * (size_t)nnode, 0.0);
    for (int i = 0; i < ncell; ++i) {
        const int32_t *cn = m.cone + (size_t)cells[i] * nv;
        double mid[3] = {0.0, 0.0, 0.0};
        for (int v = 0; v < nv; ++v)
            for (int d = 0; d < 3; ++d) mid[d] += m.coords[3 * (size_t)cn[v] + d] / nv;
        for (int b = 0; b < nb; ++b) {
            const int32_t g = cl[(size_t)i * nb + b] = rank[m.closure[(size_t)cells[i] * nb + b]];
            for (int d = 0; d < 3; ++d) x[3 * (size_t)g + d] += mid[d];
            ++ptr[g + 1];
        }
    }
    for (int i = 0; i < nnode; ++i) {
        for (int d = 0; d < 3; ++d) x[3 * (size_t)i + d] /= ptr[i + 1];
        ptr[i + 1] += ptr[i];
    }
    inc.resize(ptr[nnode]);
    {
        std::vector<int32_t> fill(ptr.begin(), ptr.end() - 1);
        for (int i = 0; i < ncell; ++i)
            for (int b = 0; b < nb; ++b) inc[fill[cl[(size_t)i * nb + b]]++] = i;
    }
    // as many tiles as allowed (the work of a tile is what a call waits for), not below 32 nodes each
    const int parts = std::max(1, std::min(max_tiles, nnode / 32));
    std::vector<int32_t> order(nnode), sizes;
    std::iota(order.begin(), order.end(), 0);
    bisect_equal(x, order.data(), (int)order.size(), parts, sizes);
    const TileLimits lim = tile_limits(nb == 8 ? 1 : 2);
    gp->tile_cell_ptr.assign(1, 0);
    gp->tile_node_ptr.assign(1, 0);
    gp->tile_vert_ptr.assign(1, 0);
    sizes.erase(std::remove(sizes.begin(), sizes.end(), 0), sizes.end());
    std::vector<int32_t> first(1, 0);
    for (int32_t sz : sizes) first.push_back(first.back() + sz);
    struct Tile {
        std::vector<int32_t> cells, nodes, verts;
        std::vector<uint16_t> lcl, lcn;  // [cells][nb], [cells][nv]
    };
    std::vector<Tile> tiles(sizes.size());
    parallel_ranges((int)tiles.size(), [&](int lo, int hi) {
        // the tile that last saw each node and cell, and the node's place in it
        std::vector<int32_t> seen(nnode, -1), place(nnode), cell_seen(ncell, -1), tc, own;
        std::vector<uint64_t> used;
        std::vector<std::pair<int, int>> by;
        for (int t = lo; t < hi; ++t) {
            Tile &T = tiles[t];
            std::vector<int32_t> &tn = T.nodes, &tv = T.verts;
            // the tile's nodes, its cells, and the other nodes and the vertices of those
            tn.assign(order.begin() + first[t], order.begin() + first[t + 1]);
            std::sort(tn.begin(), tn.end());
            own = tn;
            tc.clear();
            for (int32_t i : own) {
                seen[i] = t;
                for (int k = ptr[i]; k < ptr[i + 1]; ++k)
                    if (cell_seen[inc[k]] != t) {
                        cell_seen[inc[k]] = t;
                        tc.push_back(inc[k]);
                    }
            }
            if ((int)tc.size() > kGatherCells) {  // too large (found out below)
                T.cells = tc;
                continue;
            }
            std::sort(tc.begin(), tc.end());
            for (int32_t c : tc)
                for (int b = 0; b < nb; ++b) {
                    const int32_t g = cl[(size_t)c * nb + b];
                    if (seen[g] != t) {
                        seen[g] = t;
                        tn.push_back(g);
                    }
                }
            std::sort(tn.begin() + own.size(), tn.end());
            for (size_t k = 0; k < tn.size(); ++k) place[tn[k]] = (int32_t)k;
            if (!m.cone_is_closure) {
                for (int32_t c : tc)
                    tv.insert(tv.end(), m.cone + (size_t)cells[c] * nv, m.cone + (size_t)(cells[c] + 1) * nv);
                distinct(tv);
            }
            // tets sorted by colour, so that a wave's atomic targets are mostly distinct (hexes keep mesh order:
            // neighbouring lanes, spread banks)
            by.clear();
            used.assign(tn.size(), 0);
            for (size_t i = 0; i < tc.size(); ++i) {
                int k = 0;
                if (nb != 8) {
                    uint64_t mask = 0;
                    for (int b = 0; b < nb; ++b) mask |= used[place[cl[(size_t)tc[i] * nb + b]]];
                    while (k < 63 && ((mask >> k) & 1)) ++k;
                    for (int b = 0; b < nb; ++b) used[place[cl[(size_t)tc[i] * nb + b]]] |= (uint64_t)1 << k;
                }
                by.emplace_back(k, (int)i);
            }
            std::sort(by.begin(), by.end());
            T.cells.reserve(tc.size());
            T.lcl.reserve(tc.size() * nb);
            T.lcn.reserve(m.cone_is_closure ? 0 : tc.size() * nv);
            for (const auto &e : by) {
                const int32_t c = tc[e.second];
                T.cells.push_back(cells[c]);
                for (int b = 0; b < nb; ++b) T.lcl.push_back((uint16_t)place[cl[(size_t)c * nb + b]]);
                for (int b = 0; b < nv && !m.cone_is_closure; ++b)
                    T.lcn.push_back((uint16_t)place_of(tv, m.cone[(size_t)cells[c] * nv + b]));
            }
            for (int32_t &g : tn) g = nodes[g];
        }
    });
    for (size_t t = 0; t < tiles.size(); ++t) {
        const Tile &T = tiles[t];
        if ((int)T.cells.size() > kGatherCells || (int)T.nodes.size() > lim.nodes || (int)T.verts.size() > lim.verts) {
            *gp = HostPlan();
            return 0;
        }
        gp->cells.insert(gp->cells.end(), T.cells.begin(), T.cells.end());
        gp->tile_nodes.insert(gp->tile_nodes.end(), T.nodes.begin(), T.nodes.end());
        gp->tile_verts.insert(gp->tile_verts.end(), T.verts.begin(), T.verts.end());
        gp->tile_cell_ptr.push_back((int32_t)gp->cells.size());
        gp->tile_node_ptr.push_back((int32_t)gp->tile_nodes.size());
        gp->tile_vert_ptr.push_back((int32_t)gp->tile_verts.size());
        gp->tile_nown.push_back(sizes[t]);
        gp->tile_halo_off.push_back(0);
        gp->tile_ncolor.push_back(1);
        gp->max_nodes = std::max(gp->max_nodes, (int)T.nodes.size());
        gp->max_verts = std::max(gp->max_verts, (int)T.verts.size());
    }
    gp->num_tiles = (int)gp->tile_nown.size();
    const size_t n = gp->cells.size();
    gp->color.assign(n, 0);
    gp->lclosure.resize(nb * n);
    gp->lcone.resize(nv * n);
    for (int t = 0; t < gp->num_tiles; ++t)
        for (int i = gp->tile_cell_ptr[t]; i < gp->tile_cell_ptr[t + 1]; ++i) {
            const size_t k = (size_t)(i - gp->tile_cell_ptr[t]);
            for (int b = 0; b < nb; ++b) gp->lclosure[(size_t)b * n + i] = tiles[t].lcl[k * nb + b];
            if (!m.cone_is_closure)
                for (int b = 0; b < nv; ++b) gp->lcone[(size_t)b * n + i] = tiles[t].lcn[k * nv + b];
        }
    if (m.cone_is_closure) {
        gp->tile_verts = gp->tile_nodes;
        gp->tile_vert_ptr = gp->tile_node_ptr;
        gp->lcone = gp->lclosure;
        gp->max_verts = gp->max_nodes;
    }
    *fits = true;
    return 0;
}

}  // namespace plx
