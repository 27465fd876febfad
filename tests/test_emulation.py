"""CPU checks of the gfx950 kernels' indexing and element math: the host emulation of the tile
kernels (same plan, LDS staging, colour phases, halo reduction and element code, every index
bounds-checked) against the oracle.  No GPU."""
import ctypes
import os

import numpy as np
import pytest

from pylith_amd import _lib as L
from pylith_amd import meshgen as mg
from pylith_amd import meshio_ascii
from general_meshes import delaunay_p2

GOLDEN = os.path.join(os.path.dirname(__file__), "golden")


def emulate(m, aux, u, label=0, scalar=L.FP64, mode=L.INSERT_VALUES, r0=None, algo=L.ALGO_AUTO):
    lib = L.load()
    mu, K = aux[:, 1], aux[:, 2]
    lam_mu = np.ascontiguousarray(np.stack([K - 2 * mu / 3, mu], 1))
    dt = np.float64 if scalar == L.FP64 else np.float32
    uu = np.ascontiguousarray(u, dt)
    r = np.zeros_like(uu) if r0 is None else np.ascontiguousarray(r0, dt).copy()
    i32 = lambda a: np.ascontiguousarray(a, np.int32)
    cl, co, lb = i32(m.closure), i32(m.cone), i32(m.labels)
    xy = np.ascontiguousarray(m.coords, np.float64)
    err = lib.plx_debug_emulate_apply(m.cell_type, m.num_cells, m.num_vertices, m.num_nodes,
                                      cl.ctypes.data_as(L._i32p), co.ctypes.data_as(L._i32p),
                                      xy.ctypes.data_as(L._dblp), lb.ctypes.data_as(L._i32p), label,
                                      lam_mu.ctypes.data_as(L._dblp), scalar,
                                      ctypes.c_void_p(uu.ctypes.data), ctypes.c_void_p(r.ctypes.data), mode, algo)
    assert err == 0, f"emulation error {err}"
    return r


def relerr(a, b):
    return float(np.abs(a - b).max() / np.abs(b).max())


def cases():
    ref, _ = meshio_ascii.read(os.path.join(GOLDEN, "hex.mesh"))
    pert = mg.hex_box((9, 7, 5), (0, 0, 0), (900.0, 700.0, 500.0), ordered=False)
    rng = np.random.default_rng(11)
    x = pert.coords.copy()
    inner = np.all((x > 1) & (x < np.array([899, 699, 499])), axis=1)
    x[inner] += rng.uniform(-25, 25, (inner.sum(), 3))
    pert.coords = pert.node_coords = x
    return {
        "hex16": (mg.hex_box(16, (0, 0, 0), (6000.0, 6000.0, 6000.0)), 0),
        "hex_ragged": (mg.hex_box((13, 3, 2), (0, 0, 0), (13.0, 3.0, 2.0)), 0),
        "hex_unordered_nonaffine": (pert, 0),
        "hex_ref_fixture": (ref, 24),
        "tet8": (mg.tet_p2_box(8, (0, 0, 0), (6000.0, 6000.0, 6000.0)), 0),
        "tet_unordered": (mg.tet_p2_box((3, 4, 2), (0, 0, 0), (3.0, 4.0, 2.0), ordered=False), 0),
        # numbering without locality: the planner tiles these in Morton order
        "hex_renumbered": (mg.renumbered(mg.hex_box(12, (0, 0, 0), (1200.0, 1200.0, 1200.0)), 7), 0),
        "tet_renumbered": (mg.renumbered(mg.tet_p2_box(6, (0, 0, 0), (600.0, 600.0, 600.0)), 8), 0),
    }


@pytest.mark.parametrize("algo", [L.ALGO_QUADRATURE_POINTS, L.ALGO_FACTORED])
@pytest.mark.parametrize("name", list(cases()))
def test_emulated_kernels_match_oracle(oracle, name, algo):
    m, label = cases()[name]
    aux, sizes = mg.elastic_aux(m.num_cells, seed=5, vs_sigma=0.2, vp_vs=1.8)
    u = mg.random_field(m.num_nodes, 3)
    ref = oracle.Problem(m, aux, sizes).residual(u, 1)
    r = emulate(m, aux, u, label, algo=algo)
    assert relerr(r, ref) <= 1e-12
    r32 = emulate(m, aux, u, label, scalar=L.FP32, algo=algo)
    assert relerr(r32.astype(np.float64), ref) <= 2e-5
    radd = emulate(m, aux, u, label, mode=L.ADD_VALUES, r0=np.ones_like(u), algo=algo)
    assert relerr(radd - 1.0, ref) <= 1e-11


EMULATE_PAIRS = 100


def pair_cases():
    one = mg.tet_p2_box(1, (0, 0, 0), (1.0, 1.0, 1.0))
    single = mg.Mesh(one.cell_type, one.closure[:1], one.cone[:1], one.coords, one.node_coords, one.shape,
                     one.labels[:1])
    big = mg.tet_p2_box((9, 7, 8), (0, 0, 0), (900.0, 700.0, 800.0))
    big.labels = (np.random.default_rng(3).random(big.num_cells) < 0.6).astype(np.int32)  # scattered cells
    return {
        "one_cell": (single, 0),                                            # a cell without a partner
        "one_cube": (one, 0),
        "tet8": (mg.tet_p2_box(8, (0, 0, 0), (6000.0, 6000.0, 6000.0)), 0),  # several tiles
        "tet_odd": (mg.tet_p2_box((5, 3, 1), (0, 0, 0), (5.0, 3.0, 1.0), ordered=False), 0),
        "tet_slab": (mg.tet_p2_box((31, 2, 2), (0, 0, 0), (31.0, 2.0, 2.0)), 0),
        "tet_renumbered": (mg.renumbered(mg.tet_p2_box(7, (0, 0, 0), (600.0, 600.0, 600.0)), 8), 0),
        "tet_label": (big, 1),
    }


def general_pair_case(name):
    """Meshes whose cells do not all find a partner: nearly full tiles with more than kPairTilePairs pairs and
    lone cells are cut again."""
    if name == "label_95":
        m = mg.tet_p2_box((27, 29, 31), (0, 0, 0), (2700.0, 2900.0, 3100.0))
        m.labels = (np.random.default_rng(2).random(m.num_cells) < 0.95).astype(np.int32)
        return m, 1
    return (delaunay_p2(12500, 1) if name == "delaunay" else delaunay_p2(3000, 4, jitter=0.45)), 0


@pytest.mark.parametrize("name", ["delaunay", "delaunay_jitter", "label_95"])
def test_emulated_pair_kernel_on_general_meshes(name):
    """As above; det J of the Delaunay cells carries a relative error of a few eps / 0.02, some 1e-14, in either
    kernel (the vertices enter in another order): 1e-12."""
    m, label = general_pair_case(name)
    aux, _ = mg.elastic_aux(m.num_cells, seed=5, vs_sigma=0.2, vp_vs=1.8)
    u = mg.random_field(m.num_nodes, 3)
    ref = emulate(m, aux, u, label)
    assert relerr(emulate(m, aux, u, label, algo=EMULATE_PAIRS), ref) <= 1e-12
    r32 = emulate(m, aux, u, label, scalar=L.FP32, algo=EMULATE_PAIRS)
    assert relerr(r32.astype(np.float64), ref) <= 2e-5


@pytest.mark.parametrize("name", list(pair_cases()))
def test_emulated_pair_kernel_matches_tile_kernel(name):
    """The pair plan and kernel against the tile kernel's emulation (itself held to the oracle above):
    the same sums in another order."""
    m, label = pair_cases()[name]
    aux, _ = mg.elastic_aux(m.num_cells, seed=5, vs_sigma=0.2, vp_vs=1.8)
    u = mg.random_field(m.num_nodes, 3)
    ref = emulate(m, aux, u, label)
    assert relerr(emulate(m, aux, u, label, algo=EMULATE_PAIRS), ref) <= 1e-13
    r32 = emulate(m, aux, u, label, scalar=L.FP32, algo=EMULATE_PAIRS)
    assert relerr(r32.astype(np.float64), ref) <= 2e-5
    radd = emulate(m, aux, u, label, mode=L.ADD_VALUES, r0=np.ones_like(u), algo=EMULATE_PAIRS)
    assert relerr(radd - 1.0, ref) <= 1e-11


@pytest.mark.parametrize("split", ["edges", "all"])
def test_emulated_pair_kernel_with_nodes_split_on_a_plane(split):
    """Cells on either side of a plane share its vertices' coordinates (cone) but not its nodes (closure):
    all of them, or those of its edges alone.  Faces there do not make pairs."""
    m = mg.tet_p2_box((4, 3, 2), (0, 0, 0), (4.0, 3.0, 2.0))
    far = m.node_coords[m.closure].mean(1)[:, 0] > 2.0
    plane = np.flatnonzero(np.abs(m.node_coords[:, 0] - 2.0) < 1e-9)
    if split == "edges":
        plane = np.setdiff1d(plane, m.closure[:, :4])
    new = np.arange(m.num_nodes)
    new[plane] = m.num_nodes + np.arange(len(plane))
    m.closure[far] = new[m.closure[far]]
    m.node_coords = np.concatenate([m.node_coords, m.node_coords[plane]])
    aux, _ = mg.elastic_aux(m.num_cells, seed=5, vs_sigma=0.2, vp_vs=1.8)
    u = mg.random_field(m.num_nodes, 3)
    ref = emulate(m, aux, u)
    for algo in (EMULATE_PAIRS, EMULATE_GATHER):
        assert relerr(emulate(m, aux, u, algo=algo), ref) <= 1e-13


@pytest.mark.parametrize("algo", [L.ALGO_FACTORED, EMULATE_PAIRS])
@pytest.mark.parametrize("h", [1e-14, 1e-11, 1e-8, 1.0, 1e6, 1e9])
def test_emulated_fp32_p2_element_over_lengths(algo, h):
    """FP32 with moduli of rock and cells of any length: the products stay inside FP32's range while
    mu det J does (1e10 h^3 from 1e-32 to 1e37 here)."""
    m = mg.tet_p2_box((4, 3, 2), (0, 0, 0), (4 * h, 3 * h, 2 * h))
    aux, _ = mg.elastic_aux(m.num_cells, seed=5, vs_sigma=0.2, vp_vs=1.8)
    u = 1e3 * h * mg.random_field(m.num_nodes, 3)
    ref = emulate(m, aux, u)
    r32 = emulate(m, aux, u, scalar=L.FP32, algo=algo)
    assert relerr(r32.astype(np.float64), ref) <= 2e-5


EMULATE_GATHER = 101  # PLX_EMULATE_GATHER


def gather_cases():
    big = mg.tet_p2_box(6, (0, 0, 0), (1.0, 1.0, 1.0))
    big.labels = (np.arange(big.num_cells) % 3 == 0).astype(np.int32)
    return {
        "one_hex": (mg.hex_box(1, (0, 0, 0), (1.0, 1.0, 1.0)), 0),
        "one_cube": (mg.tet_p2_box(1, (0, 0, 0), (1.0, 1.0, 1.0)), 0),
        "tet_label": (big, 1),  # nodes of the mesh outside the key
        "hex_max": (mg.hex_box(38, (0, 0, 0), (1.0, 1.0, 1.0)), 0),  # about the largest that fits 512 tiles
        "tet_large": (mg.tet_p2_box(16, (0, 0, 0), (1.0, 1.0, 1.0)), 0),
        # (on a random mesh det J carries a few eps / 0.02: see the pair kernel's)
        "delaunay_jitter": (delaunay_p2(1000, 4, jitter=0.3, min_quality=0.1), 0),
        **cases(),
    }


@pytest.mark.parametrize("name", list(gather_cases()))
def test_emulated_gather_plan_matches_tile_plan(name):
    """The tile kernel over the gather plan against the tile plan's emulation: the same sums in another
    order (rounding of at most some 24 additions per node in FP64, of the element products in FP32)."""
    m, label = gather_cases()[name]
    aux, _ = mg.elastic_aux(m.num_cells, seed=5, vs_sigma=0.2, vp_vs=1.8)
    u = mg.random_field(m.num_nodes, 3)
    ref = emulate(m, aux, u, label)
    assert relerr(emulate(m, aux, u, label, algo=EMULATE_GATHER), ref) <= 1e-13
    r32 = emulate(m, aux, u, label, scalar=L.FP32, algo=EMULATE_GATHER)
    assert relerr(r32.astype(np.float64), ref) <= 2e-5
    radd = emulate(m, aux, u, label, mode=L.ADD_VALUES, r0=np.ones_like(u), algo=EMULATE_GATHER)
    assert relerr(radd - 1.0, ref) <= 1e-11
