// Host memory running out while the plans are made: every allocation in turn (in strides) fails once.
// The planners must either throw std::bad_alloc to their caller or return; an exception that leaves one of
// their threads, or joinable threads left behind, would end the process.
// usage: plan_alloc <num> -- box of num^3 x 6 P2 tetrahedra or num^3 hexes
#include <atomic>
#include <cstdio>
#include <cstdlib>
#include <new>

#include "plx_plan.hpp"

static std::atomic<long> g_left{-1}, g_count{0};

void *operator new(size_t n) {
    g_count.fetch_add(1, std::memory_order_relaxed);
    if (g_left.load(std::memory_order_relaxed) >= 0 && g_left.fetch_sub(1) == 0) throw std::bad_alloc();
    if (void *p = std::malloc(n ? n : 1)) return p;
    throw std::bad_alloc();
}
void operator delete(void *p) noexcept { std::free(p); }
void operator delete(void *p, size_t) noexcept { std::free(p); }

using namespace plx;

struct Box {
    std::vector<int32_t> closure, cone;
    std::vector<double> coords;
    int nodes = 0, verts = 0;
};

static Box hexes(int n) {
    Box b;
    const int w = n + 1;
    auto id = [&](int i, int j, int k) { return (k * w + j) * w + i; };
    for (int k = 0; k < n; ++k)
        for (int j = 0; j < n; ++j)
            for (int i = 0; i < n; ++i)
                for (int v : {id(i, j, k), id(i + 1, j, k), id(i + 1, j + 1, k), id(i, j + 1, k), id(i, j, k + 1),
                              id(i + 1, j, k + 1), id(i + 1, j + 1, k + 1), id(i, j + 1, k + 1)})
                    b.closure.push_back(v);
    for (int k = 0; k < w; ++k)
        for (int j = 0; j < w; ++j)
            for (int i = 0; i < w; ++i)
                for (int x : {i, j, k}) b.coords.push_back(x);
    b.cone = b.closure;
    b.nodes = b.verts = w * w * w;
    return b;
}

// Each cube in six tetrahedra along its diagonal; nodes at the half-grid points.
static Box tets(int n) {
    Box b;
    const int w = n + 1, h = 2 * n + 1;
    const int path[6][2] = {{0, 1}, {1, 2}, {2, 0}, {1, 0}, {2, 1}, {0, 2}};
    for (int k = 0; k < n; ++k)
        for (int j = 0; j < n; ++j)
            for (int i = 0; i < n; ++i)
                for (int t = 0; t < 6; ++t) {
                    int p[4][3] = {{i, j, k}, {i, j, k}, {i, j, k}, {i + 1, j + 1, k + 1}};
                    p[1][path[t][0]]++;
                    p[2][path[t][0]]++;
                    p[2][path[t][1]]++;
                    if (t >= 3) std::swap(p[1], p[2]);  // (orientation)
                    const int e[10][2] = {{0, 0}, {1, 1}, {2, 2}, {3, 3}, {0, 1}, {0, 2}, {0, 3}, {1, 2}, {1, 3}, {2, 3}};
                    for (auto &q : e)
                        b.closure.push_back(((p[q[0]][2] + p[q[1]][2]) * h + p[q[0]][1] + p[q[1]][1]) * h + p[q[0]][0] + p[q[1]][0]);
                    for (auto &v : p) b.cone.push_back((v[2] * w + v[1]) * w + v[0]);
                }
    for (int k = 0; k < w; ++k)
        for (int j = 0; j < w; ++j)
            for (int i = 0; i < w; ++i)
                for (int x : {i, j, k}) b.coords.push_back(x);
    b.verts = w * w * w;
    b.nodes = h * h * h;
    return b;
}

template <typename F>
static int fail_in_turn(const char *name, const F &work) {
    g_count = 0;
    work();
    const long total = g_count;
    int thrown = 0;
    for (long k = 0; k < total; k += 1 + total / 60) {
        g_left = k;
        try {
            work();
        } catch (const std::bad_alloc &) {
            ++thrown;
        }
        g_left = -1;
    }
    std::printf("%s: %ld allocations, %d failures reached the caller\n", name, total, thrown);
    std::fflush(stdout);
    return thrown > 0 ? 0 : 1;
}

int main(int argc, char **argv) {
    const int n = argc > 1 ? std::atoi(argv[1]) : 10;
    int bad = 0;
    for (int hex = 0; hex < 2; ++hex) {
        const Box b = hex ? hexes(n) : tets(n);
        const int nb = hex ? 8 : 10, nv = hex ? 8 : 4;
        const MeshView mv{nb, nv, (int)b.closure.size() / nb, b.nodes, b.verts, b.closure.data(), b.cone.data(),
                          nullptr, hex == 1, b.coords.data()};
        TileLimits lim = tile_limits(hex ? 1 : 2);
        lim.cells = 32;  // (many tiles: several threads)
        HostPlan base;
        std::string err;
        if (build_host_plan(mv, 0, lim, &base, &err)) return 2;
        bad += fail_in_turn("tile plan", [&] {
            HostPlan hp;
            std::string e;
            (void)build_host_plan(mv, 0, lim, &hp, &e);
        });
        bad += fail_in_turn("gather plan", [&] {
            HostPlan gp;
            bool fits = false;
            (void)build_gather_plan(mv, base, 512, &gp, &fits);
        });
        if (!hex)
            bad += fail_in_turn("pair plan", [&] {
                PairPlan pp;
                std::string e;
                (void)build_pair_plan(mv, base, &pp, &e);
            });
    }
    return bad;
}
