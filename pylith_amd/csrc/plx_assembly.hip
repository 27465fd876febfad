// plx_assembly.hip -- gfx950 kernels of the residual / Jacobian-action apply.
//
// One persistent workgroup walks a sequence of tiles of cells (one or two cells, or a pair, per thread):
//   1. the tile's nodal field and vertex coordinates are staged in LDS through the tile's
//      node / vertex lists (coalesced where node numbers run contiguously); the next tile's
//      gathers are issued into registers before the current tile's arithmetic;
//   2. each thread evaluates its element vectors (Q1 hex: sum-factorized 2x2x2 Gauss or the
//      modal form on affine cells; P2 tet: 14-point rule or its P1-moment form) from the
//      device twin of the pointwise kernel;
//   3. element vectors are accumulated into an LDS node buffer either colour by colour (fixed
//      summation order, bitwise reproducible) or with LDS atomic adds into an FP64 accumulator
//      (the default; the order of the additions into one node, and so the last bits, may vary);
//   4. nodes owned by the tile are written straight to the output vector; shared nodes leave
//      as partial sums in the halo buffer, reduced in slot order by a node-ordered second kernel.
//      Small meshes take a gather plan instead: overlapping tiles that own nodes, and no halo.
// No global atomics are used.
#include <algorithm>
#include <map>
#include <mutex>

#include "plx_element.hpp"
#include "plx_internal.hpp"
#include "plx_plan.hpp"
#include "plx_reduce.hpp"

namespace plx {

// Reference tables of the P2 element in constant memory (each device holds its own copy).
__constant__ P2Tables c_p2;
constexpr int kMaxDevices = 64;
static bool g_tables_ready[kMaxDevices] = {};
static std::mutex g_device_mu;

struct DevTab {
    __device__ static double w(int q) { return c_p2.w[q]; }
    __device__ static double dphi(int q, int b, int k) { return c_p2.dphi[q][b][k]; }
    __device__ static double lam(int q, int v) { return c_p2.lam[q][v]; }
};

// Called with the DM's device current (plx_dm_create).
static int ensure_tables(plx_dm dm) {
    std::lock_guard<std::mutex> lock(g_device_mu);
    if (g_tables_ready[dm->device]) return 0;
    P2Tables t;
    p2_fill_tables(&t);
    PLX_HIP(dm, hipMemcpyToSymbol(HIP_SYMBOL(c_p2), &t, sizeof(t)));
    g_tables_ready[dm->device] = true;
    return 0;
}

// --------------------------------------------------------------------------------------------
// Scratch of the allocation-free residual entry point (plx_compute_residual_noalloc): the
// shared-node partial sums of one apply live in this file-scope device array instead of the
// key's own halo buffer.  Each device holds its own copy until the process ends; host code
// reaches it only through the address hipGetSymbolAddress returns on that device (the array's
// name is a host-side stand-in).  Every call on one device shares the array, so calls that
// overlap on one device race.  The apply writes every halo slot before the reduction reads it,
// so nothing needs clearing between calls.
// --------------------------------------------------------------------------------------------
constexpr size_t kScratchBytes = (size_t)64 << 20;
static __device__ __align__(256) unsigned char scratch[kScratchBytes];
static void *g_scratch_ptr[kMaxDevices] = {};

int device_setup(plx_dm dm) {
    int dev = 0;
    PLX_HIP(dm, hipGetDevice(&dev));
    if (dev < 0 || dev >= kMaxDevices) return set_error(dm, 1, "device index beyond the supported range");
    dm->device = dev;
    {
        std::lock_guard<std::mutex> lock(g_device_mu);
        if (!g_scratch_ptr[dev]) {
            void *p = nullptr;
            PLX_HIP(dm, hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
            if (!p) return set_error(dm, 76, "scratch array has no device address");
            g_scratch_ptr[dev] = p;
        }
    }
    return ensure_tables(dm);
}

// --------------------------------------------------------------------------------------------
// Tile kernel.
// --------------------------------------------------------------------------------------------
struct ApplyArgs {
    TilePlanDev p;
    const uint8_t *color;   // [stride] colour of each key cell (tile-local greedy colouring)
    const void *mat;        // [2][stride] lambda, mu
    const void *u;
    void *r;
    void *halo;
    int mode;
    double scale;           // multiplies the element vectors (e.g. -1 for the SPD operator -J)
    const int32_t *heads;      // TileHead of the tiles this launch covers, in order
    int num_list;
    const void *records;       // packed 16-bit local closure (+ cone) per key cell
    const double *prestress;   // Q1: per-point stress added to sigma, [6][8][stride] (nullptr: none)
    P2Scale p2;
};

// Cell solution values read from the tile's LDS buffer (component c, local basis b).
template <typename Real, int NB>
struct LdsAcc {
    const Real *sU;
    int lc[NB];
    __device__ __forceinline__ Real operator()(int c, int b) const { return sU[3 * lc[b] + c]; }
};
template <typename Real>
struct LdsAccQ1 {
    const Real *sU;
    int lc[8];
    __device__ __forceinline__ Real operator()(int c, int l) const { return sU[3 * lc[q1_lex(l)] + c]; }
};

constexpr int kAccColored = 0, kAccAtomic = 1;

// Tile extents (TileHead), loaded one word per lane two tiles ahead and read from the lanes when the
// tile's ids go out.  Read in place, each tile began with a wait for its extents that also waited for
// the previous tile's stores (loads and stores complete in order): 137 -> 128 us on 153 x 149 x 157
// hexes.
__device__ __forceinline__ int head_word(const int32_t *heads, int tile) { return heads[8 * (size_t)tile + (threadIdx.x & 7)]; }
__device__ __forceinline__ TileHead head_of(int word) {
    TileHead h;
    h.c0 = __builtin_amdgcn_readlane(word, 0);
    h.nc = __builtin_amdgcn_readlane(word, 1);
    h.n0 = __builtin_amdgcn_readlane(word, 2);
    h.nn = __builtin_amdgcn_readlane(word, 3);
    h.v0 = __builtin_amdgcn_readlane(word, 4);
    h.nvt = __builtin_amdgcn_readlane(word, 5);
    h.nown = __builtin_amdgcn_readlane(word, 6);
    h.hoff = __builtin_amdgcn_readlane(word, 7);
    return h;
}

// A tile's node sums to the output: owned nodes to their rows (the ids in gn), shared ones to the
// halo slots.  All of a thread's sums are read before the first is stored.
template <typename Real, typename Acc, int SLOTS, int NT>
__device__ __forceinline__ void write_out(const Acc *sR, const int (&gn)[SLOTS], int nn, int nown, int hoff, int tid,
                                          Real *r, Real *halo, bool insert) {
    Real w[SLOTS][3];
#pragma unroll
    for (int j = 0; j < SLOTS; ++j) {
        const int k = min(tid + j * NT, nn - 1);
#pragma unroll
        for (int c = 0; c < 3; ++c) w[j][c] = (Real)sR[3 * k + c];
    }
#pragma unroll
    for (int j = 0; j < SLOTS; ++j) {
        const int k = tid + j * NT;
        if (k < nn) {
            Real *dst = k < nown ? r + 3 * (size_t)gn[j] : halo + 3 * ((size_t)hoff + (size_t)(k - nown));
            if (!insert && k < nown) {
#pragma unroll
                for (int c = 0; c < 3; ++c) w[j][c] += dst[c];
            }
#pragma unroll
            for (int c = 0; c < 3; ++c) dst[c] = w[j][c];
        }
    }
}

// Map slot i to a tile so that each of the 8 XCDs (round-robin workgroup dispatch) walks a
// contiguous range of tiles: neighbouring tiles then share that XCD's L2.
__device__ __forceinline__ int xcd_tile(int i, int n) {
    const int per = n >> 3, rem = n & 7;
    const int x = i & 7, j = i >> 3;
    return x * per + min(x, rem) + j;
}

// Workgroup shape per cell type and vector type: NT threads, CPT cells per thread, PFN node
// slots and PFV vertex slots per thread for the register prefetch of the next tile.
template <int CT, typename Real>
struct Shape;
template <typename Real>
struct Shape<PLX_HEX_Q1, Real> {
    // RECW: uint4 words per cell record (8 x uint16 closure)
    static constexpr int NT = 256, CPT = 2, NB = 8, NV = 8, PFN = 3, PFV = 0, RECW = 1;
};
// P2: 4-wave workgroups over the 384-cell tile (cells 0-255 on the first pass, 256-383 on the
// second), two workgroups per CU at the FP64 kernel's register count (2 waves per SIMD).  One cell
// per thread in 6-wave workgroups measured slower (63 x 66 x 61 x 6 cells, FP64: 92 us, 96 us with
// the registers cut to three waves per SIMD, against 80 us on the same build; 76 us now).
// record: 10 x uint16 closure, 4 x uint16 cone, 2 padding = 2 uint4 words
template <typename Real>
struct Shape<PLX_TET_P2, Real> {
    static constexpr int NT = 256, CPT = 2, NB = 10, NV = 4, PFN = 3, PFV = 1, RECW = 2;
};

// Entry k of a packed 16-bit cell record.
template <int W>
__device__ __forceinline__ int rec_get(const uint4 (&r)[W], int k) {
    const uint4 &w = r[k >> 3];
    const int h = (k >> 1) & 3;
    const unsigned v = h == 0 ? w.x : h == 1 ? w.y : h == 2 ? w.z : w.w;
    return (k & 1) ? (int)(v >> 16) : (int)(v & 0xffffu);
}

// One tile's data on its way from HBM: gathered node values and coordinates, the cells' local
// closures, moduli and colours (registers).  The gathers go out in two phases: the node / vertex ids
// before the previous tile's cells, whose arithmetic hides their latency, and the values at them later.
// Every load is unconditional, at positions clamped into the tile: slots past its end repeat its last
// entry.  (A branch around each load keeps its destination registers alive around the loop: 30 to 60
// registers, and with them the spills of the Q1 quadrature-point kernels.)
template <typename Real, int CT>
struct Stage {
    using S = Shape<CT, Real>;
    int c0, nc, ncolor, n0, nn, v0, nvt, nown, hoff;
    int gn[S::PFN];                          // node ids (the write-out uses them again)
    int gv[CT == PLX_HEX_Q1 ? 1 : S::PFV];   // P2 vertex ids
    Real pu[S::PFN][3];
    double px[CT == PLX_HEX_Q1 ? S::PFN : S::PFV][3];
    uint4 rec[S::CPT][S::RECW];  // packed 16-bit local closure (and cone) of each cell
    Real lam[S::CPT], mu[S::CPT];
    int color[S::CPT];
    __device__ __forceinline__ void extents(const TileHead &h) {
        c0 = h.c0;
        nc = h.nc & 0xffff;
        ncolor = h.nc >> 16;
        n0 = h.n0;
        nn = h.nn;
        v0 = h.v0;
        nvt = h.nvt;
        nown = h.nown;
        hoff = h.hoff;
    }
};

template <typename Real, int CT>
__device__ __forceinline__ void fetch_ids(Stage<Real, CT> &T, const ApplyArgs &A, const TileHead &h, int tid) {
    using S = Shape<CT, Real>;
    T.extents(h);
#pragma unroll
    for (int j = 0; j < S::PFN; ++j) T.gn[j] = A.p.tile_nodes[h.n0 + min(tid + j * S::NT, h.nn - 1)];
    if constexpr (CT != PLX_HEX_Q1) T.gv[0] = A.p.tile_verts[h.v0 + min(tid, h.nvt - 1)];
}

template <typename Real, int CT, int ACC>
__device__ __forceinline__ void fetch_cells(Stage<Real, CT> &T, const ApplyArgs &A, int tid) {
    using S = Shape<CT, Real>;
    const Real *mat = static_cast<const Real *>(A.mat);
    const uint4 *recs = reinterpret_cast<const uint4 *>(A.records);
#pragma unroll
    for (int i = 0; i < S::CPT; ++i) {
        const int pos = T.c0 + min(tid + i * S::NT, T.nc - 1);
#pragma unroll
        for (int w = 0; w < S::RECW; ++w) T.rec[i][w] = recs[(size_t)pos * S::RECW + w];
        // unscaled here (scaled where used): the fetch then has no use of these loads to wait for
        T.lam[i] = mat[pos];
        T.mu[i] = mat[A.p.stride + pos];
        if (ACC == kAccColored) T.color[i] = A.color[pos];
    }
}

template <typename Real, int CT>
__device__ __forceinline__ void fetch_values(Stage<Real, CT> &T, const ApplyArgs &A) {
    using S = Shape<CT, Real>;
    const Real *u = static_cast<const Real *>(A.u);
    const double *coords = A.p.coords;
#pragma unroll
    for (int j = 0; j < S::PFN; ++j) {
        const size_t g = (size_t)T.gn[j];
#pragma unroll
        for (int c = 0; c < 3; ++c) T.pu[j][c] = u[3 * g + c];
        if constexpr (CT == PLX_HEX_Q1) {
#pragma unroll
            for (int d = 0; d < 3; ++d) T.px[j][d] = coords[3 * g + d];
        }
    }
    if constexpr (CT != PLX_HEX_Q1) {
#pragma unroll
        for (int d = 0; d < 3; ++d) T.px[0][d] = coords[3 * (size_t)T.gv[0] + d];
    }
}

// LDS of a tile kernel: nodal values, the accumulator and coordinates at fixed places (the addresses
// then differ by constants), sized for every thread's slots.
template <typename Real, int CT, typename Acc>
constexpr size_t tile_lds_bytes() {
    using S = Shape<CT, Real>;
    return (size_t)S::PFN * S::NT * 3 * (sizeof(Real) + sizeof(Acc)) +
           (size_t)(CT == PLX_HEX_Q1 ? S::PFN * S::NT : S::PFV * S::NT) * 3 * sizeof(double);
}

// Element paths of the tile kernel: the factorized form (kernels linear in the gradient with
// per-cell coefficients, affine cells), the quadrature-point form on affine cells, and the
// quadrature-point form on any Q1 cell (P2 tets are affine: their quadrature-point form is
// kPathQpAffine).
enum { kPathFactored = 0, kPathQpAffine = 1, kPathQpGeneral = 2 };

// Persistent, software-pipelined tile kernel: each workgroup walks its slots; while it works
// on one tile, the gathers of its next tile are in flight.
template <typename Real, int CT, int PATH, int ACC, int MINW>
__global__ void __launch_bounds__((Shape<CT, Real>::NT), MINW) apply_tiles(ApplyArgs A) {
    using S = Shape<CT, Real>;
    constexpr int NT = S::NT, NB = S::NB, NV = S::NV;
    static_assert(S::PFN * NT >= 768 && S::CPT * NT >= (CT == PLX_HEX_Q1 ? 512 : 384), "tile limits");
    static_assert(CT == PLX_HEX_Q1 || (S::PFV == 1 && NT >= 192), "vertex limit");
    extern __shared__ __align__(16) unsigned char smem[];
    const int tid = threadIdx.x;
    const int G = gridDim.x;
    int slot = blockIdx.x;
    if (slot >= A.num_list) return;
    auto word_of = [&](int s) { return head_word(A.heads, xcd_tile(s, A.num_list)); };
    Stage<Real, CT> cur;
    int next_word = slot + G < A.num_list ? word_of(slot + G) : 0;
    fetch_ids<Real, CT>(cur, A, head_of(word_of(slot)), tid);
    fetch_cells<Real, CT, ACC>(cur, A, tid);
    fetch_values<Real, CT>(cur, A);
    Real *r = static_cast<Real *>(A.r);
    Real *halo = static_cast<Real *>(A.halo);
    const bool insert = A.mode == PLX_INSERT_VALUES;
    // LDS atomics accumulate in FP64 whatever the vector type (native ds_add_f64; FP32 calls
    // round once at the write-out)
    using Acc = typename std::conditional<ACC == kAccAtomic, double, Real>::type;
    Acc *sR = reinterpret_cast<Acc *>(smem);
    Real *sU = reinterpret_cast<Real *>(sR + 3 * S::PFN * NT);
    double *sX = reinterpret_cast<double *>(sU + 3 * S::PFN * NT);
    constexpr bool DIRECT = CT != PLX_HEX_Q1 && PATH == kPathFactored && ACC == kAccAtomic;
    // The next tile's node values go out between the thread's two cells and arrive during the second
    // (153 x 149 x 157 hexes, factored: 128 us; after both cells 146 us).  The Q1 quadrature-point
    // kernels, whose elements fill the registers, load them and the cells' data after both (80 x 71 x 66
    // non-affine hexes: 44.5 us, 45.6 us between the cells).
    constexpr bool LATE = CT == PLX_HEX_Q1 && PATH != kPathFactored;
    while (true) {
#pragma unroll
        for (int j = 0; j < S::PFN; ++j) {
            const int k = tid + j * NT;
#pragma unroll
            for (int c = 0; c < 3; ++c) {
                sU[3 * k + c] = cur.pu[j][c];
                sR[3 * k + c] = Acc(0);
            }
            if constexpr (CT == PLX_HEX_Q1) {
#pragma unroll
                for (int d = 0; d < 3; ++d) sX[3 * k + d] = cur.px[j][d];
            }
        }
        if constexpr (CT != PLX_HEX_Q1) {
#pragma unroll
            for (int d = 0; d < 3; ++d) sX[3 * tid + d] = cur.px[0][d];
        }
        __syncthreads();

        const int next_slot = slot + G;
        const bool has_next = next_slot < A.num_list;
        Stage<Real, CT> nxt;
        // the next tile's loads are issued at a raised wave priority, so the SIMD issues them
        // ahead of the arithmetic of its other waves (P2 FP64 kernel -1.3 %; the write-out below
        // at priority 1: Q1 -1.4 %)
        __builtin_amdgcn_s_setprio(2);
        if (has_next) {
            const TileHead h = head_of(next_word);
            if (next_slot + G < A.num_list) next_word = word_of(next_slot + G);
            fetch_ids<Real, CT>(nxt, A, h, tid);
            if constexpr (!LATE) fetch_cells<Real, CT, ACC>(nxt, A, tid);
        }
        __builtin_amdgcn_s_setprio(0);

#pragma unroll
        for (int i = 0; i < S::CPT; ++i) {
            const bool active = tid + i * NT < cur.nc;
            int lc[NB];
#pragma unroll
            for (int b = 0; b < NB; ++b) lc[b] = rec_get(cur.rec[i], b);
            Real re[3][NB];
            if (active) {
                const Real lam = (Real)A.scale * cur.lam[i], mu = (Real)A.scale * cur.mu[i];
                if constexpr (CT == PLX_HEX_Q1) {
                    Real rl[3][8];
                    const LdsAccQ1<double> xacc{sX, {lc[0], lc[1], lc[2], lc[3], lc[4], lc[5], lc[6], lc[7]}};
                    const LdsAccQ1<Real> acc{sU, {lc[0], lc[1], lc[2], lc[3], lc[4], lc[5], lc[6], lc[7]}};
                    if constexpr (PATH == kPathFactored) {
                        // affine tiles only (the plan routes other tiles to the quadrature-point kernel)
                        double J[9];
                        q1_affine_jacobian(xacc, J);
                        q1_element_affine<Real>(J, acc, lam, mu, rl);
                    } else {
                        const double *pre = A.prestress ? A.prestress + cur.c0 + tid + i * NT : nullptr;
                        q1_element_qp<Real, PATH == kPathQpAffine>(xacc, acc, lam, mu, rl, pre, (size_t)A.p.stride,
                                                                   (Real)A.scale);
                    }
#pragma unroll
                    for (int l = 0; l < 8; ++l)
#pragma unroll
                        for (int c = 0; c < 3; ++c) re[c][q1_lex(l)] = rl[c][l];
                } else {
                    double X[4][3];
#pragma unroll
                    for (int v = 0; v < NV; ++v) {
                        const int lv = rec_get(cur.rec[i], NB + v);
#pragma unroll
                        for (int d = 0; d < 3; ++d) X[v][d] = sX[3 * lv + d];
                    }
                    if constexpr (PATH == kPathFactored) {
                        const LdsAcc<Real, 10> acc{sU, {lc[0], lc[1], lc[2], lc[3], lc[4], lc[5], lc[6], lc[7], lc[8], lc[9]}};
                        // LDS atomics take an entry as soon as it is formed
                        p2_element_linear<Real>(X, acc, lam, mu, A.p2, [&](int c, int b, Real v) {
                            if constexpr (DIRECT) atomicAdd(&sR[3 * lc[b] + c], (Acc)v);
                            else re[c][b] = v;
                        });
                    } else {
                        Real U[3][10];
#pragma unroll
                        for (int b = 0; b < NB; ++b)
#pragma unroll
                            for (int c = 0; c < 3; ++c) U[c][b] = sU[3 * lc[b] + c];
                        p2_element<Real, DevTab>(X, U, lam, mu, re);
                    }
                }
            }
            if constexpr (ACC == kAccAtomic) {
                // LDS atomics: no colour phases; the order of the additions into a node varies
                if (!DIRECT && active) {
#pragma unroll
                    for (int b = 0; b < NB; ++b)
#pragma unroll
                        for (int c = 0; c < 3; ++c) atomicAdd(&sR[3 * lc[b] + c], (Acc)re[c][b]);
                }
            } else {
                // cells of one colour share no node: fixed summation order (cells i = 0 of the
                // workgroup colour by colour, then cells i = 1), reproducible bits
                for (int col = 0; col < cur.ncolor; ++col) {
                    __syncthreads();
                    if (active && cur.color[i] == col) {
#pragma unroll
                        for (int b = 0; b < NB; ++b)
#pragma unroll
                            for (int c = 0; c < 3; ++c) sR[3 * lc[b] + c] += re[c][b];
                    }
                }
            }
            if (!LATE && i == 0 && has_next) {
                __builtin_amdgcn_s_setprio(2);
                fetch_values<Real, CT>(nxt, A);
                __builtin_amdgcn_s_setprio(0);
            }
        }
        __syncthreads();
        __builtin_amdgcn_s_setprio(1);
        if (LATE && has_next) {
            fetch_cells<Real, CT, ACC>(nxt, A, tid);
            fetch_values<Real, CT>(nxt, A);
        }
        // a gather plan (no halo) has nothing to store for the nodes that other tiles own
        write_out<Real, Acc, S::PFN, NT>(sR, cur.gn, halo ? cur.nn : cur.nown, cur.nown, cur.hoff, tid, r, halo, insert);
        __builtin_amdgcn_s_setprio(0);
        if (!has_next) break;
        __syncthreads();  // every read of this tile's LDS precedes the next tile's staging
        cur = nxt;
        slot = next_slot;
    }
}

// --------------------------------------------------------------------------------------------
// P2 pair kernel: the factored residual / action with LDS atomics, one pair of face-sharing cells per
// thread (PairPlan).  A pair reads 14 nodes and 5 vertices from LDS and adds to 14 nodes where two
// cells take 20, 8 and 20, its record is 24 bytes where theirs are 64, and 512-cell tiles leave fewer
// shared nodes.  63 x 66 x 61 x 6 cells, profiler: 73.6 us and 19.5 us for the halo sums against 75.9 and 21.2 us for
// the tile kernel (FP32, 40 x 44 x 37 x 6: 17.8 against 19.2 us).
// The tile kernel above is bound on chip (63 x 66 x 61 x 6 cells, before its extents were fetched two tiles ahead and
// its loads made unconditional: 80 us, 68 us with every gather served from L2, 57 us without its atomics,
// 42 us without the element): LDS accesses are what pairing cuts.  Same pipeline, with everything but the next tile's ids after the cells: two cells at
// once leave no registers for it (between the two halves of the element: 79 us against 74).
// --------------------------------------------------------------------------------------------
struct PairArgs {
    int num_tiles;
    const int32_t *heads, *nodes, *verts;
    const uint2 *rec;   // [pairs][3]
    const void *mat;    // [pairs][4] lambda, mu of the two cells
    const double *coords;
    const void *u;
    void *r, *halo;
    int mode;
    float area;    // P2Scale
    double scale;  // with P2Scale's factor
};

constexpr int kPairThreads = 256, kPairSlots = kPairTileNodes / kPairThreads;
static_assert(kPairThreads == kPairTilePairs && kPairThreads >= kPairTileVerts, "one pair and one vertex per thread");

template <typename Real>
constexpr size_t pair_lds_bytes() {
    return (size_t)kPairTileNodes * 3 * (sizeof(double) + sizeof(Real)) + (size_t)kPairTileVerts * 3 * sizeof(double);
}

template <typename Real>
struct PairStage {
    int p0, np, nn, nown, hoff;
    int gn[kPairSlots], gv;
    Real pu[kPairSlots][3];
    double px[3];
    uint2 rec[3];
    Real mat[4];
};

// Every load is unconditional, at positions clamped into the tile: slots past its end repeat its last
// entry (a branch around each load keeps its destination registers alive around the loop).
template <typename Real>
__device__ __forceinline__ void pair_fetch_ids(PairStage<Real> &T, const PairArgs &A, const TileHead &h, int tid) {
    T.p0 = h.c0;
    T.np = h.nc;
    T.nn = h.nn;
    T.nown = h.nown;
    T.hoff = h.hoff;
#pragma unroll
    for (int j = 0; j < kPairSlots; ++j) T.gn[j] = A.nodes[h.n0 + min(tid + j * kPairThreads, h.nn - 1)];
    T.gv = A.verts[h.v0 + min(tid, h.nvt - 1)];
}

template <typename Real>
__device__ __forceinline__ void pair_fetch_values(PairStage<Real> &T, const PairArgs &A, int tid) {
    const Real *u = static_cast<const Real *>(A.u);
    const size_t p = (size_t)T.p0 + (size_t)min(tid, T.np - 1);
#pragma unroll
    for (int w = 0; w < 3; ++w) T.rec[w] = A.rec[3 * p + w];
    const Real *m = static_cast<const Real *>(A.mat) + 4 * p;
#pragma unroll
    for (int i = 0; i < 4; ++i) T.mat[i] = m[i];
#pragma unroll
    for (int j = 0; j < kPairSlots; ++j)
#pragma unroll
        for (int c = 0; c < 3; ++c) T.pu[j][c] = u[3 * (size_t)T.gn[j] + c];
#pragma unroll
    for (int d = 0; d < 3; ++d) T.px[d] = A.coords[3 * (size_t)T.gv + d];
}

template <typename Real>
__global__ void __launch_bounds__(kPairThreads, 2) apply_pairs(PairArgs A) {
    extern __shared__ __align__(16) unsigned char smem[];
    double *sR = reinterpret_cast<double *>(smem);
    double *sX = sR + 3 * kPairTileNodes;
    Real *sU = reinterpret_cast<Real *>(sX + 3 * kPairTileVerts);
    const int tid = threadIdx.x;
    const int G = gridDim.x;
    int slot = blockIdx.x;
    if (slot >= A.num_tiles) return;
    PairStage<Real> cur;
    auto word_of = [&](int s) { return head_word(A.heads, xcd_tile(s, A.num_tiles)); };
    int next_word = slot + G < A.num_tiles ? word_of(slot + G) : 0;
    pair_fetch_ids<Real>(cur, A, head_of(word_of(slot)), tid);
    pair_fetch_values<Real>(cur, A, tid);
    Real *r = static_cast<Real *>(A.r);
    Real *halo = static_cast<Real *>(A.halo);
    const bool insert = A.mode == PLX_INSERT_VALUES;
    while (true) {
#pragma unroll
        for (int j = 0; j < kPairSlots; ++j) {
            const int k = tid + j * kPairThreads;
#pragma unroll
            for (int c = 0; c < 3; ++c) {
                sU[3 * k + c] = cur.pu[j][c];
                sR[3 * k + c] = 0.0;
            }
        }
#pragma unroll
        for (int d = 0; d < 3; ++d) sX[3 * tid + d] = cur.px[d];
        __syncthreads();
        const int next_slot = slot + G;
        const bool has_next = next_slot < A.num_tiles;
        PairStage<Real> nxt;
        // the next tile's loads at a raised wave priority, ahead of the other waves' arithmetic
        __builtin_amdgcn_s_setprio(2);
        if (has_next) {
            const TileHead h = head_of(next_word);
            if (next_slot + G < A.num_tiles) next_word = word_of(next_slot + G);
            pair_fetch_ids<Real>(nxt, A, h, tid);
        }
        __builtin_amdgcn_s_setprio(0);
        if (tid < cur.np) {
            int n[14];
            Real AA[9], AB[9], SA[4][6], SB[4][6];
            Real qa, qb;
            {
                const unsigned w[6] = {cur.rec[0].x, cur.rec[0].y, cur.rec[1].x, cur.rec[1].y, cur.rec[2].x, cur.rec[2].y};
#pragma unroll
                for (int j = 0; j < 12; ++j) n[j] = (int)((w[j / 3] >> (10 * (j % 3))) & 1023u);
                n[12] = (int)(w[4] & 1023u);
                n[13] = (int)((w[4] >> 10) & 1023u);
                double X[5][3];
#pragma unroll
                for (int v = 0; v < 5; ++v) {
                    const int lv = v < 4 ? (int)((w[5] >> (8 * v)) & 255u) : (int)((w[4] >> 20) & 255u);
#pragma unroll
                    for (int d = 0; d < 3; ++d) X[v][d] = sX[3 * lv + d];
                }
                qa = p2_geometry<Real>(X, A.scale, A.area, AA);
                const double XB[4][3] = {{X[4][0], X[4][1], X[4][2]}, {X[1][0], X[1][1], X[1][2]},
                                         {X[3][0], X[3][1], X[3][2]}, {X[2][0], X[2][1], X[2][2]}};
                qb = p2_geometry<Real>(XB, A.scale, A.area, AB);
            }
            p2_pair_strains<sizeof(Real) == 8, Real>([&](int c, int j) { return sU[3 * n[j] + c]; }, AA, AB, SA, SB);
            p2_vertex_stresses<Real>(qa, cur.mat[0], cur.mat[1], SA);
            p2_vertex_stresses<Real>(qb, cur.mat[2], cur.mat[3], SB);
            p2_pair_contract<sizeof(Real) == 8, Real>(
                SA, SB, AA, AB, [&](int c, int j, Real v) { atomicAdd(&sR[3 * n[j] + c], (double)v); });
        }
        __syncthreads();
        __builtin_amdgcn_s_setprio(1);
        if (has_next) pair_fetch_values<Real>(nxt, A, tid);
        write_out<Real, double, kPairSlots, kPairThreads>(sR, cur.gn, cur.nn, cur.nown, cur.hoff, tid, r, halo, insert);
        __builtin_amdgcn_s_setprio(0);
        if (!has_next) break;
        __syncthreads();  // every read of this tile's LDS precedes the next tile's staging
        cur = nxt;
        slot = next_slot;
    }
}

// --------------------------------------------------------------------------------------------
// The apply of a CG iteration over a gather plan, with the direction update before it and the mask and
// the dot product after it (CgArgs): an iteration is this kernel and the solver's cg_step.  One tile and
// at most one cell per thread in a workgroup.  Every tile forms the direction at all its nodes, the same
// way, from z and the old direction; owners store it, into a buffer of its own, since other tiles still
// read the old one.  At 10,000s of dofs each kernel is launch and latency: 24 x 22 x 25 hexes, FP32
// point-block Jacobi: 18 us an iteration in four kernels, 14 us in two.
// --------------------------------------------------------------------------------------------
template <typename Real, int CT>
__global__ void __launch_bounds__((Shape<CT, Real>::NT), 2) cg_apply(ApplyArgs A, CgArgs C) {
    using S = Shape<CT, Real>;
    constexpr int NT = S::NT, NB = S::NB, NV = S::NV;
    static_assert(kGatherCells <= NT && NT == 256, "one cell per thread, 256-thread reductions");
    extern __shared__ __align__(16) unsigned char smem[];
    __shared__ double s[4];
    const int tid = threadIdx.x;
    double *sR = reinterpret_cast<double *>(smem);
    Real *sU = reinterpret_cast<Real *>(sR + 3 * S::PFN * NT);
    double *sX = reinterpret_cast<double *>(sU + 3 * S::PFN * NT);
    Stage<Real, CT> T;
    fetch_ids<Real, CT>(T, A, head_of(head_word(A.heads, xcd_tile(blockIdx.x, A.num_list))), tid);
    const int pos = T.c0 + min(tid, T.nc - 1);
    uint4 rec[S::RECW];
#pragma unroll
    for (int w = 0; w < S::RECW; ++w) rec[w] = reinterpret_cast<const uint4 *>(A.records)[(size_t)pos * S::RECW + w];
    const Real lam = (Real)A.scale * static_cast<const Real *>(A.mat)[pos];
    const Real mu = (Real)A.scale * static_cast<const Real *>(A.mat)[A.p.stride + pos];
    // every load goes out before the sum below is waited for; a tile's nodes mostly fit the first slot
    const Real *u = static_cast<const Real *>(A.u), *z = static_cast<const Real *>(C.z);
    Real pv[S::PFN][3] = {};
    Real zv[S::PFN][3] = {};
    uint8_t fx[S::PFN] = {};
#pragma unroll
    for (int j = 0; j < S::PFN; ++j)
        if (j * NT < T.nn) {
            const size_t g = (size_t)T.gn[j];
            fx[j] = C.fixed[g];
#pragma unroll
            for (int c = 0; c < 3; ++c) {
                pv[j][c] = u[3 * g + c];
                zv[j][c] = z[3 * g + c];
                if constexpr (CT == PLX_HEX_Q1) T.px[j][c] = A.p.coords[3 * g + c];
            }
        }
    if constexpr (CT != PLX_HEX_Q1) {
#pragma unroll
        for (int d = 0; d < 3; ++d) T.px[0][d] = A.p.coords[3 * (size_t)T.gv[0] + d];
    }
    const double old = *C.rz_old, rz = total(C.part_rz, C.nblk, s);
    const Real beta = (Real)(old != 0.0 ? rz / old : 0.0);
    if (blockIdx.x == 0 && tid == 0) *C.rz = rz;
    Real *pout = static_cast<Real *>(C.p_out), *r = static_cast<Real *>(A.r);
#pragma unroll
    for (int j = 0; j < S::PFN; ++j)
        if (j * NT < T.nn) {
            const int k = tid + j * NT;
#pragma unroll
            for (int c = 0; c < 3; ++c) {
                zv[j][c] += beta * pv[j][c];
                sU[3 * k + c] = zv[j][c];
                sR[3 * k + c] = 0.0;
                if constexpr (CT == PLX_HEX_Q1) sX[3 * k + c] = T.px[j][c];
            }
        }
    if constexpr (CT != PLX_HEX_Q1) {
#pragma unroll
        for (int d = 0; d < 3; ++d) sX[3 * tid + d] = T.px[0][d];
    }
    __syncthreads();
    if (tid < T.nc) {
        int lc[NB];
#pragma unroll
        for (int b = 0; b < NB; ++b) lc[b] = rec_get(rec, b);
        if constexpr (CT == PLX_HEX_Q1) {
            const LdsAccQ1<double> xacc{sX, {lc[0], lc[1], lc[2], lc[3], lc[4], lc[5], lc[6], lc[7]}};
            const LdsAccQ1<Real> acc{sU, {lc[0], lc[1], lc[2], lc[3], lc[4], lc[5], lc[6], lc[7]}};
            double J[9];
            Real rl[3][8];
            q1_affine_jacobian(xacc, J);
            q1_element_affine<Real>(J, acc, lam, mu, rl);
#pragma unroll
            for (int l = 0; l < 8; ++l)
#pragma unroll
                for (int c = 0; c < 3; ++c) atomicAdd(&sR[3 * lc[q1_lex(l)] + c], (double)rl[c][l]);
        } else {
            double X[4][3];
#pragma unroll
            for (int v = 0; v < NV; ++v) {
                const int lv = rec_get(rec, NB + v);
#pragma unroll
                for (int d = 0; d < 3; ++d) X[v][d] = sX[3 * lv + d];
            }
            const LdsAcc<Real, 10> acc{sU, {lc[0], lc[1], lc[2], lc[3], lc[4], lc[5], lc[6], lc[7], lc[8], lc[9]}};
            p2_element_linear<Real>(X, acc, lam, mu, A.p2, [&](int c, int b, Real v) { atomicAdd(&sR[3 * lc[b] + c], (double)v); });
        }
    }
    __syncthreads();
    double pq = 0.0;
#pragma unroll
    for (int j = 0; j < S::PFN; ++j) {
        const int k = tid + j * NT;
        if (k < T.nown) {
#pragma unroll
            for (int c = 0; c < 3; ++c) {
                const Real q = (fx[j] >> c) & 1 ? Real(0) : (Real)sR[3 * k + c];
                r[3 * (size_t)T.gn[j] + c] = q;
                pout[3 * (size_t)T.gn[j] + c] = zv[j][c];
                pq += (double)zv[j][c] * (double)q;
            }
        }
    }
    pq = block_sum(pq, s);
    if (tid == 0) C.part_pq[blockIdx.x] = pq;
}

// Shared nodes: sum the tiles' partials in tile order.
template <typename Real>
__global__ void __launch_bounds__(256) reduce_halo(int nshared, const int32_t *__restrict__ node,
                                                   const int32_t *__restrict__ ptr,
                                                   const int32_t *__restrict__ slot,
                                                   const Real *__restrict__ halo, Real *r, int mode) {
    const int s = blockIdx.x * blockDim.x + threadIdx.x;
    if (s >= nshared) return;
    const int j0 = ptr[s], j1 = ptr[s + 1];
    const size_t g = 3 * (size_t)node[s];
    Real a0 = Real(0), a1 = Real(0), a2 = Real(0);
    // slots four at a time: their ids, then their values, then the sums in slot order (the
    // ids are read at clamped positions inside this node's range; extra lanes are not summed)
    for (int jb = j0; jb < j1; jb += 4) {
        int sl[4];
#pragma unroll
        for (int q = 0; q < 4; ++q) sl[q] = slot[min(jb + q, j1 - 1)];
        Real v[4][3];
#pragma unroll
        for (int q = 0; q < 4; ++q)
#pragma unroll
            for (int c = 0; c < 3; ++c) v[q][c] = halo[3 * (size_t)sl[q] + c];
#pragma unroll
        for (int q = 0; q < 4; ++q)
            if (jb + q < j1) {
                a0 += v[q][0];
                a1 += v[q][1];
                a2 += v[q][2];
            }
    }
    if (mode == PLX_INSERT_VALUES) {
        r[g + 0] = a0;
        r[g + 1] = a1;
        r[g + 2] = a2;
    } else {
        r[g + 0] += a0;
        r[g + 1] += a1;
        r[g + 2] += a2;
    }
}

static TilePlanDev plan_dev(plx_dm dm, const KeyPlan *kp) {
    TilePlanDev p;
    p.num_tiles = kp->num_tiles;
    p.stride = (int)kp->cells.size();
    p.tile_cell_ptr = kp->d_tile_cell_ptr;
    p.tile_node_ptr = kp->d_tile_node_ptr;
    p.tile_nown = kp->d_tile_nown;
    p.tile_nodes = kp->d_tile_nodes;
    p.tile_vert_ptr = kp->d_tile_vert_ptr;
    p.tile_verts = kp->d_tile_verts;
    p.tile_halo_off = kp->d_tile_halo_off;
    p.lclosure = kp->d_lclosure;
    p.lcone = kp->d_lcone;
    p.coords = dm->d_coords;
    return p;
}

// Resident workgroups per CU of a persistent tile kernel at this LDS size, from the occupancy
// calculator (registers, LDS and waves), cached per kernel and size; at most 4.
static int resident_per_cu(const void *kernel, int nt, size_t lds, int fallback) {
    static std::mutex mu;
    static std::map<std::pair<const void *, size_t>, int> cache;
    std::lock_guard<std::mutex> lock(mu);
    const auto key = std::make_pair(kernel, lds);
    const auto it = cache.find(key);
    if (it != cache.end()) return it->second;
    int n = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, kernel, nt, lds) != hipSuccess || n < 1) n = fallback;
    n = std::min(n, 4);
    cache[key] = n;
    return n;
}

template <typename Real>
static int reduce_shared(plx_dm dm, int n, const int32_t *node, const int32_t *ptr, const int32_t *slot,
                         const void *halo, void *r, int mode, bool log) {
    if (n == 0) return 0;
    ScopedEvent ev(dm, log ? "plx:reduce_halo" : nullptr);
    hipLaunchKernelGGL(reduce_halo<Real>, dim3((n + 255) / 256), dim3(256), 0, dm->stream, n, node, ptr, slot,
                       static_cast<const Real *>(halo), static_cast<Real *>(r), mode);
    PLX_HIP(dm, hipGetLastError());
    return 0;
}

bool takes_pairs(plx_dm dm, const KeyPlan *kp) {
    return kp->pairs.num_tiles > 0 && kp->pairs.d_mat64 && dm->algorithm != PLX_ALGO_QUADRATURE_POINTS &&
           dm->accumulate != PLX_ACCUMULATE_COLORED && dm->min_waves <= 2;
}

// (a gather plan is made only where it is the faster one: make_second_plans)
bool takes_gather(plx_dm dm, const KeyPlan *kp) {
    return kp->gather.num_tiles > 0 && kp->gather.d_mat64 && dm->algorithm != PLX_ALGO_QUADRATURE_POINTS &&
           dm->accumulate != PLX_ACCUMULATE_COLORED;
}

template <typename Real>
static int apply_pairs_typed(plx_dm dm, KeyPlan *kp, const void *u, void *r, int mode, double scale, void *halo,
                             bool log, bool reduce) {
    const PairDev &P = kp->pairs;
    PairArgs A;
    A.num_tiles = P.num_tiles;
    A.heads = P.d_heads;
    A.nodes = P.d_nodes;
    A.verts = P.d_verts;
    A.rec = reinterpret_cast<const uint2 *>(P.d_records);
    A.mat = std::is_same<Real, double>::value ? (const void *)P.d_mat64 : (const void *)P.d_mat32;
    A.coords = dm->d_coords;
    A.u = u;
    A.r = r;
    A.halo = halo ? halo : kp->d_halo;
    A.mode = mode;
    A.area = dm->p2_scale.area;
    A.scale = std::is_same<Real, double>::value ? scale : scale * dm->p2_scale.factor;
    if (dm->num_cu <= 0) PLX_HIP(dm, hipDeviceGetAttribute(&dm->num_cu, hipDeviceAttributeMultiprocessorCount, 0));
    const size_t lds = pair_lds_bytes<Real>();
    const int per_cu = resident_per_cu(reinterpret_cast<const void *>(&apply_pairs<Real>), kPairThreads, lds, 2);
    const int resident = ((std::max(dm->num_cu, 8) * per_cu + 7) / 8) * 8;
    {
        ScopedEvent ev(dm, log ? "plx:apply_tiles" : nullptr);
        hipLaunchKernelGGL(apply_pairs<Real>, dim3(std::min(P.num_tiles, resident)), dim3(kPairThreads), lds, dm->stream, A);
    }
    PLX_HIP(dm, hipGetLastError());
    if (!reduce) return 0;
    return reduce_shared<Real>(dm, P.num_shared, P.d_shared_node, P.d_shared_ptr, P.d_shared_slot, A.halo, r, mode, log);
}

template <typename Real>
static int apply_typed(plx_dm dm, KeyPlan *kp, const void *u, void *r, int mode, double scale,
                       const double *prestress, void *halo, bool log, bool reduce) {
    if (!prestress && takes_pairs(dm, kp)) return apply_pairs_typed<Real>(dm, kp, u, r, mode, scale, halo, log, reduce);
    ApplyArgs A;
    A.scale = scale;
    A.p2 = dm->p2_scale;
    A.prestress = prestress;
    A.p = plan_dev(dm, kp);
    A.color = kp->d_color;
    A.mat = std::is_same<Real, double>::value ? (const void *)kp->d_mat64 : (const void *)kp->d_mat32;
    A.u = u;
    A.r = r;
    A.halo = halo ? halo : kp->d_halo;
    A.mode = mode;
    A.records = kp->d_records;
    int n_affine = kp->num_tiles_affine, n_tiles = kp->num_tiles;
    const int32_t *affine = kp->d_heads_affine, *tiles = kp->d_heads;
    const bool gather = !prestress && takes_gather(dm, kp);
    if (gather) {
        const GatherDev &G = kp->gather;
        n_affine = n_tiles = G.num_tiles;  // a Q1 key with a gather plan has affine tiles only
        affine = tiles = G.d_heads;
        A.p.tile_nodes = G.d_nodes;
        A.p.tile_verts = G.d_verts;
        A.p.stride = (int)G.cells.size();
        A.mat = std::is_same<Real, double>::value ? (const void *)G.d_mat64 : (const void *)G.d_mat32;
        A.records = G.d_records;
        A.halo = nullptr;
    }
    // a per-point prestress needs the quadrature-point path
    const bool linear = dm->algorithm != PLX_ALGO_QUADRATURE_POINTS && !prestress;
    // AUTO: LDS atomics (FP64 accumulator, native ds_add_f64) for both vector types
    const bool atomic = dm->accumulate != PLX_ACCUMULATE_COLORED;
    // persistent grid: as many workgroups per CU as the kernel's registers and LDS let reside
    // (a multiple of 8 in all keeps each workgroup on the XCD whose tile range it walks), never
    // more than there are tiles
    if (dm->num_cu <= 0) PLX_HIP(dm, hipDeviceGetAttribute(&dm->num_cu, hipDeviceAttributeMultiprocessorCount, 0));
    const int ncu = std::max(dm->num_cu, 8);
    {
    ScopedEvent ev(dm, log ? "plx:apply_tiles" : nullptr);
#define PLX_LAUNCH_W(CT, PATH, ACC, W, N)                                                             \
    do {                                                                                             \
        const void *kfn = reinterpret_cast<const void *>(&apply_tiles<Real, CT, PATH, ACC, W>);       \
        constexpr size_t lds =                                                                       \
            tile_lds_bytes<Real, CT, typename std::conditional<ACC == kAccAtomic, double, Real>::type>(); \
        const int per_cu = resident_per_cu(kfn, Shape<CT, Real>::NT, lds, dm->wg_per_cu);            \
        const int resident = ((ncu * per_cu + 7) / 8) * 8;                                           \
        hipLaunchKernelGGL((apply_tiles<Real, CT, PATH, ACC, W>), dim3(std::min(N, resident)),         \
                           dim3(Shape<CT, Real>::NT), lds, dm->stream, A);                           \
    } while (0)
#define PLX_LAUNCH(CT, PATH, ACC, LIST, N)                                                           \
    do {                                                                                             \
        A.heads = LIST;                                                                              \
        A.num_list = N;                                                                              \
        if (N > 0) {                                                                                 \
            if (minw <= 2) PLX_LAUNCH_W(CT, PATH, ACC, 2, N);                                          \
            else if (minw == 3) PLX_LAUNCH_W(CT, PATH, ACC, 3, N);                                     \
            else PLX_LAUNCH_W(CT, PATH, ACC, 4, N);                                                    \
        }                                                                                            \
    } while (0)
    const int minw = dm->min_waves;
    if (dm->cell_type == PLX_HEX_Q1) {
        // affine tiles: the factorized kernel (or the quadrature-point one on affine cells); the
        // rest: the quadrature-point kernel with the Jacobian at each point
        if (linear) {
            if (atomic) {
                PLX_LAUNCH(PLX_HEX_Q1, kPathFactored, kAccAtomic, affine, n_affine);
                PLX_LAUNCH(PLX_HEX_Q1, kPathQpGeneral, kAccAtomic, kp->d_heads_general, kp->num_tiles_general);
            } else {
                PLX_LAUNCH(PLX_HEX_Q1, kPathFactored, kAccColored, affine, n_affine);
                PLX_LAUNCH(PLX_HEX_Q1, kPathQpGeneral, kAccColored, kp->d_heads_general, kp->num_tiles_general);
            }
        } else {
            if (atomic) {
                PLX_LAUNCH(PLX_HEX_Q1, kPathQpAffine, kAccAtomic, affine, n_affine);
                PLX_LAUNCH(PLX_HEX_Q1, kPathQpGeneral, kAccAtomic, kp->d_heads_general, kp->num_tiles_general);
            } else {
                PLX_LAUNCH(PLX_HEX_Q1, kPathQpAffine, kAccColored, affine, n_affine);
                PLX_LAUNCH(PLX_HEX_Q1, kPathQpGeneral, kAccColored, kp->d_heads_general, kp->num_tiles_general);
            }
        }
    } else {
        if (linear) {
            if (atomic) PLX_LAUNCH(PLX_TET_P2, kPathFactored, kAccAtomic, tiles, n_tiles);
            else PLX_LAUNCH(PLX_TET_P2, kPathFactored, kAccColored, tiles, n_tiles);
        } else {
            if (atomic) PLX_LAUNCH(PLX_TET_P2, kPathQpAffine, kAccAtomic, tiles, n_tiles);
            else PLX_LAUNCH(PLX_TET_P2, kPathQpAffine, kAccColored, tiles, n_tiles);
        }
    }
#undef PLX_LAUNCH_W
#undef PLX_LAUNCH
    }
    PLX_HIP(dm, hipGetLastError());
    if (!reduce || gather) return 0;
    return reduce_shared<Real>(dm, kp->num_shared, kp->d_shared_node, kp->d_shared_ptr, kp->d_shared_slot, A.halo, r, mode,
                               log);
}

// Residual and Jacobian action share the element operator: for isotropic linear elasticity
// J v = F(v); for generalized Maxwell F(u) = J u + (the state term), with J the elastic operator
// at the effective shear modulus (the residual adds the per-point state stress).
int launch_apply(plx_dm dm, KeyPlan *kp, int scalar_type, bool jacobian, const void *u, void *r,
                 int mode, double scale, void *halo, bool log, bool reduce) {
    if (mode != PLX_ADD_VALUES && mode != PLX_INSERT_VALUES) return set_error(dm, 1, "bad insert mode");
    const double *pre = (!jacobian && kp->genmax) ? kp->d_prestress : nullptr;
    if (pre && scalar_type != PLX_FP64) return set_error(dm, 1, "the viscoelastic residual is FP64");
    if (scalar_type == PLX_FP64) return apply_typed<double>(dm, kp, u, r, mode, scale, pre, halo, log, reduce);
    if (scalar_type == PLX_FP32) return apply_typed<float>(dm, kp, u, r, mode, scale, pre, halo, log, reduce);
    return set_error(dm, 1, "bad scalar type");
}

template <typename Real>
static int cg_apply_typed(plx_dm dm, KeyPlan *kp, const void *u, void *r, double scale, const CgArgs &C) {
    const GatherDev &G = kp->gather;
    ApplyArgs A{};
    A.p = plan_dev(dm, kp);
    A.p.tile_nodes = G.d_nodes;
    A.p.tile_verts = G.d_verts;
    A.p.stride = (int)G.cells.size();
    A.mat = std::is_same<Real, double>::value ? (const void *)G.d_mat64 : (const void *)G.d_mat32;
    A.u = u;
    A.r = r;
    A.scale = scale;
    A.p2 = dm->p2_scale;
    A.heads = G.d_heads;
    A.num_list = G.num_tiles;
    A.records = G.d_records;
    {
        ScopedEvent ev(dm, "plx:apply_tiles");
        if (dm->cell_type == PLX_HEX_Q1)
            hipLaunchKernelGGL((cg_apply<Real, PLX_HEX_Q1>), dim3(G.num_tiles), dim3(Shape<PLX_HEX_Q1, Real>::NT),
                               (tile_lds_bytes<Real, PLX_HEX_Q1, double>()), dm->stream, A, C);
        else
            hipLaunchKernelGGL((cg_apply<Real, PLX_TET_P2>), dim3(G.num_tiles), dim3(Shape<PLX_TET_P2, Real>::NT),
                               (tile_lds_bytes<Real, PLX_TET_P2, double>()), dm->stream, A, C);
    }
    PLX_HIP(dm, hipGetLastError());
    return 0;
}

int launch_cg_apply(plx_dm dm, KeyPlan *kp, int scalar_type, const void *u, void *r, double scale, const CgArgs &C) {
    return scalar_type == PLX_FP64 ? cg_apply_typed<double>(dm, kp, u, r, scale, C)
                                   : cg_apply_typed<float>(dm, kp, u, r, scale, C);
}

SharedSums shared_sums(plx_dm dm, KeyPlan *kp, bool jacobian) {
    SharedSums S;
    const bool pre = !jacobian && kp->genmax && kp->d_prestress;
    if (!pre && takes_pairs(dm, kp))
        S = {kp->pairs.num_shared, kp->pairs.d_shared_node, kp->pairs.d_shared_ptr, kp->pairs.d_shared_slot, kp->d_halo};
    else if (pre || !takes_gather(dm, kp))
        S = {kp->num_shared, kp->d_shared_node, kp->d_shared_ptr, kp->d_shared_slot, kp->d_halo};
    return S;
}

// Body force / gravity load (fixed per node): r[node] += load.
template <typename Real>
__global__ void __launch_bounds__(256) add_load(int n, const int32_t *__restrict__ node,
                                                const Real *__restrict__ load, Real *r) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const size_t g = 3 * (size_t)node[i];
    r[g + 0] += load[3 * (size_t)i + 0];
    r[g + 1] += load[3 * (size_t)i + 1];
    r[g + 2] += load[3 * (size_t)i + 2];
}

int launch_add_load(plx_dm dm, KeyPlan *kp, int scalar_type, void *r) {
    const int n = kp->num_load;
    if (scalar_type == PLX_FP64)
        hipLaunchKernelGGL(add_load<double>, dim3((n + 255) / 256), dim3(256), 0, dm->stream, n,
                           kp->d_load_node, kp->d_load64, static_cast<double *>(r));
    else
        hipLaunchKernelGGL(add_load<float>, dim3((n + 255) / 256), dim3(256), 0, dm->stream, n,
                           kp->d_load_node, kp->d_load32, static_cast<float *>(r));
    PLX_HIP(dm, hipGetLastError());
    return 0;
}

// --------------------------------------------------------------------------------------------
// Point-block diagonal of J (FP64): D_b[f][g] = -sum_q w|J| [(lambda+mu) dphi_f dphi_g
//   + mu delta_fg |grad phi|^2] for isotropic C, i.e. the diagonal blocks of the element
// matrix of Jf3 = -C.  One thread per cell, global FP64 atomics (set-up path, not timed).
// --------------------------------------------------------------------------------------------
template <int CT>
__global__ void __launch_bounds__(256) pbdiag_cells(TilePlanDev P, const int32_t *cells,
                                                    const int32_t *closure, const int32_t *cone,
                                                    const double *mat, int ncells, double *blocks) {
    constexpr int NB = CT == PLX_HEX_Q1 ? 8 : 10;
    constexpr int NV = CT == PLX_HEX_Q1 ? 8 : 4;
    const int pos = blockIdx.x * blockDim.x + threadIdx.x;
    if (pos >= ncells) return;
    const int cell = cells[pos];
    const double lam = mat[pos], mu = mat[P.stride + pos];
    double X[NV][3];
#pragma unroll
    for (int v = 0; v < NV; ++v)
#pragma unroll
        for (int d = 0; d < 3; ++d) X[v][d] = P.coords[3 * (size_t)cone[(size_t)cell * NV + v] + d];
    double D[NB][6];
#pragma unroll
    for (int b = 0; b < NB; ++b)
#pragma unroll
        for (int i = 0; i < 6; ++i) D[b][i] = 0.0;
    const int nq = CT == PLX_HEX_Q1 ? 8 : kMaxQuad;
    const double g = 0.57735026918962576451;
    const double ref[8][3] = {{-1, -1, -1}, {1, -1, -1}, {1, 1, -1}, {-1, 1, -1},
                              {-1, -1, 1},  {1, -1, 1},  {1, 1, 1},  {-1, 1, 1}};
    for (int q = 0; q < nq; ++q) {
        double dphi[NB][3], J[9] = {0}, Ji[9], w;
        if constexpr (CT == PLX_HEX_Q1) {
            const double xi[3] = {(q & 1) ? g : -g, (q & 2) ? g : -g, (q & 4) ? g : -g};
            for (int b = 0; b < 8; ++b) {
                const double a0 = 1 + ref[b][0] * xi[0], a1 = 1 + ref[b][1] * xi[1], a2 = 1 + ref[b][2] * xi[2];
                dphi[b][0] = 0.125 * ref[b][0] * a1 * a2;
                dphi[b][1] = 0.125 * a0 * ref[b][1] * a2;
                dphi[b][2] = 0.125 * a0 * a1 * ref[b][2];
            }
            for (int v = 0; v < 8; ++v)
                for (int d = 0; d < 3; ++d)
                    for (int k = 0; k < 3; ++k) J[3 * d + k] += X[v][d] * dphi[v][k];
            w = 1.0;
        } else {
            for (int b = 0; b < 10; ++b)
                for (int k = 0; k < 3; ++k) dphi[b][k] = c_p2.dphi[q][b][k];
            for (int d = 0; d < 3; ++d)
                for (int k = 0; k < 3; ++k) J[3 * d + k] = X[k + 1][d] - X[0][d];
            w = c_p2.w[q];
        }
        const double wd = w * inv3(J, Ji);
        for (int b = 0; b < NB; ++b) {
            double gp[3];
            for (int d = 0; d < 3; ++d) gp[d] = dphi[b][0] * Ji[d] + dphi[b][1] * Ji[3 + d] + dphi[b][2] * Ji[6 + d];
            const double n2 = gp[0] * gp[0] + gp[1] * gp[1] + gp[2] * gp[2];
            const double lm = lam + mu;
            D[b][0] -= wd * (lm * gp[0] * gp[0] + mu * n2);
            D[b][1] -= wd * (lm * gp[1] * gp[1] + mu * n2);
            D[b][2] -= wd * (lm * gp[2] * gp[2] + mu * n2);
            D[b][3] -= wd * lm * gp[0] * gp[1];
            D[b][4] -= wd * lm * gp[1] * gp[2];
            D[b][5] -= wd * lm * gp[0] * gp[2];
        }
    }
    for (int b = 0; b < NB; ++b) {
        double *B = blocks + 9 * (size_t)closure[(size_t)cell * NB + b];
        atomicAdd(&B[0], D[b][0]);
        atomicAdd(&B[4], D[b][1]);
        atomicAdd(&B[8], D[b][2]);
        atomicAdd(&B[1], D[b][3]);
        atomicAdd(&B[3], D[b][3]);
        atomicAdd(&B[5], D[b][4]);
        atomicAdd(&B[7], D[b][4]);
        atomicAdd(&B[2], D[b][5]);
        atomicAdd(&B[6], D[b][5]);
    }
}

// Device copies of the closure and cone index (set-up kernels only), each uploaded on first use.
int ensure_mesh_indices(plx_dm dm) {
    if (!dm->d_closure) {
        PLX_HIP(dm, hipMalloc(&dm->d_closure, dm->closure.size() * sizeof(int32_t)));
        PLX_HIP(dm, hipMemcpy(dm->d_closure, dm->closure.data(), dm->closure.size() * sizeof(int32_t), hipMemcpyHostToDevice));
    }
    if (!dm->d_cone) {
        PLX_HIP(dm, hipMalloc(&dm->d_cone, dm->cone.size() * sizeof(int32_t)));
        PLX_HIP(dm, hipMemcpy(dm->d_cone, dm->cone.data(), dm->cone.size() * sizeof(int32_t), hipMemcpyHostToDevice));
    }
    return 0;
}

int launch_pbdiag(plx_dm dm, KeyPlan *kp, double *blocks) {
    const int err = ensure_mesh_indices(dm);
    if (err) return err;
    const int n = (int)kp->cells.size();
    const TilePlanDev P = plan_dev(dm, kp);
    if (dm->cell_type == PLX_HEX_Q1)
        hipLaunchKernelGGL(pbdiag_cells<PLX_HEX_Q1>, dim3((n + 255) / 256), dim3(256), 0, dm->stream, P,
                           kp->d_cells, dm->d_closure, dm->d_cone, kp->d_mat64, n, blocks);
    else
        hipLaunchKernelGGL(pbdiag_cells<PLX_TET_P2>, dim3((n + 255) / 256), dim3(256), 0, dm->stream, P,
                           kp->d_cells, dm->d_closure, dm->d_cone, kp->d_mat64, n, blocks);
    PLX_HIP(dm, hipGetLastError());
    return 0;
}

// --------------------------------------------------------------------------------------------
// Geometry validation: count cells with a non-positive Jacobian determinant at a quadrature
// point (DMPlexComputeCellGeometryFEM rejects them).
// --------------------------------------------------------------------------------------------
template <int CT>
__global__ void __launch_bounds__(256) validate_cells(int ncells, const int32_t *cone,
                                                      const double *coords, int *bad) {
    constexpr int NV = CT == PLX_HEX_Q1 ? 8 : 4;
    const int cell = blockIdx.x * blockDim.x + threadIdx.x;
    if (cell >= ncells) return;
    double X[NV][3];
    for (int v = 0; v < NV; ++v)
        for (int d = 0; d < 3; ++d) X[v][d] = coords[3 * (size_t)cone[(size_t)cell * NV + v] + d];
    double minDet = 1e300;
    if constexpr (CT == PLX_HEX_Q1) {
        const double g = 0.57735026918962576451;
        const double ref[8][3] = {{-1, -1, -1}, {1, -1, -1}, {1, 1, -1}, {-1, 1, -1},
                                  {-1, -1, 1},  {1, -1, 1},  {1, 1, 1},  {-1, 1, 1}};
        for (int q = 0; q < 8; ++q) {
            const double xi[3] = {(q & 1) ? g : -g, (q & 2) ? g : -g, (q & 4) ? g : -g};
            double J[9] = {0}, Ji[9];
            for (int b = 0; b < 8; ++b) {
                const double a0 = 1 + ref[b][0] * xi[0], a1 = 1 + ref[b][1] * xi[1], a2 = 1 + ref[b][2] * xi[2];
                const double dp[3] = {0.125 * ref[b][0] * a1 * a2, 0.125 * a0 * ref[b][1] * a2,
                                      0.125 * a0 * a1 * ref[b][2]};
                for (int d = 0; d < 3; ++d)
                    for (int k = 0; k < 3; ++k) J[3 * d + k] += X[b][d] * dp[k];
            }
            minDet = fmin(minDet, inv3(J, Ji));
        }
    } else {
        double J[9], Ji[9];
        for (int d = 0; d < 3; ++d)
            for (int k = 0; k < 3; ++k) J[3 * d + k] = X[k + 1][d] - X[0][d];
        minDet = inv3(J, Ji);
    }
    if (!(minDet > 0.0)) atomicAdd(bad, 1);
}

int validate_geometry(plx_dm dm, int *num_bad) {
    int32_t *d_cone = nullptr;
    int *d_bad = nullptr;
    PLX_HIP(dm, hipMalloc(&d_cone, dm->cone.size() * sizeof(int32_t)));
    PLX_HIP(dm, hipMemcpy(d_cone, dm->cone.data(), dm->cone.size() * sizeof(int32_t), hipMemcpyHostToDevice));
    PLX_HIP(dm, hipMalloc(&d_bad, sizeof(int)));
    PLX_HIP(dm, hipMemset(d_bad, 0, sizeof(int)));
    const int n = dm->num_cells;
    if (dm->cell_type == PLX_HEX_Q1)
        hipLaunchKernelGGL(validate_cells<PLX_HEX_Q1>, dim3((n + 255) / 256), dim3(256), 0, 0, n, d_cone, dm->d_coords, d_bad);
    else
        hipLaunchKernelGGL(validate_cells<PLX_TET_P2>, dim3((n + 255) / 256), dim3(256), 0, 0, n, d_cone, dm->d_coords, d_bad);
    PLX_HIP(dm, hipGetLastError());
    PLX_HIP(dm, hipMemcpy(num_bad, d_bad, sizeof(int), hipMemcpyDeviceToHost));
    (void)hipFree(d_cone);
    (void)hipFree(d_bad);
    return 0;
}

}  // namespace plx

using namespace plx;

extern "C" {

int plx_compute_residual_noalloc(plx_dm dm, int label_value, int part, int scalar_type, double t,
                                 const void *locX, const void *locX_t, void *locF, int mode) {
    (void)t;
    (void)locX_t;
    KeyPlan *kp = nullptr;
    if (const int e = residual_key(dm, label_value, part, locX, locF, &kp)) return e;
    if (kp->pf_residual || !kp->f1)
        return set_error(dm, 1, "PetscPointFn-form keys are not served allocation-free: use plx_compute_residual");
    if (scalar_type != PLX_FP64 && scalar_type != PLX_FP32) return set_error(dm, 1, "bad scalar type");
    // (a viscoelastic residual takes the tile plan)
    const int64_t slots = kp->genmax ? kp->halo_slots
                          : takes_pairs(dm, kp) ? kp->pairs.halo_slots
                          : takes_gather(dm, kp) ? 0 : kp->halo_slots;
    const size_t need = (size_t)slots * 3 * (scalar_type == PLX_FP64 ? sizeof(double) : sizeof(float));
    if (need > kScratchBytes)
        return set_error(dm, 1, "the key's shared-node partial sums (" + std::to_string(need) +
                                    " bytes) exceed the allocation-free scratch (" +
                                    std::to_string(kScratchBytes) + " bytes): use plx_compute_residual");
    void *scr = g_scratch_ptr[dm->device];
    if (!scr) return set_error(dm, 76, "scratch array not set up on the DM's device");
    const int err = launch_apply(dm, kp, scalar_type, false, locX, locF, mode, 1.0, scr, false);
    if (err || kp->num_load == 0) return err;
    return launch_add_load(dm, kp, scalar_type, locF);
}

}  // extern "C"
