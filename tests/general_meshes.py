"""P2 tetrahedral meshes without the lattice structure of meshgen's boxes."""
import numpy as np

from pylith_amd import meshgen as mg

EDGES = np.array([(0, 1), (0, 2), (0, 3), (1, 2), (1, 3), (2, 3)])


def delaunay_p2(npoints, seed, jitter=None, min_quality=0.02):
    """Delaunay tetrahedra of random points in the unit cube (or of a lattice whose points are moved by up to
    `jitter` of its spacing), without the cells whose det J is below min_quality of their longest
    edge cubed: det J is then known to a few eps / min_quality."""
    from scipy.spatial import Delaunay
    rng = np.random.default_rng(seed)
    if jitter is None:
        p = rng.random((npoints, 3))
    else:
        k = round(npoints ** (1 / 3))
        g = np.stack(np.meshgrid(*[np.arange(k)] * 3, indexing="ij"), -1).reshape(-1, 3).astype(float)
        p = (g + rng.uniform(-jitter, jitter, g.shape)) / k
    t = Delaunay(p).simplices.astype(np.int64)
    det = np.linalg.det(p[t[:, 1:]] - p[t[:, :1]])
    t[det < 0] = t[det < 0][:, [0, 2, 1, 3]]
    longest = np.linalg.norm(p[t[:, EDGES[:, 0]]] - p[t[:, EDGES[:, 1]]], axis=-1).max(1)
    t = t[np.abs(det) > min_quality * longest ** 3]
    used, t = np.unique(t, return_inverse=True)
    p, t = p[used], t.reshape(-1, 4)
    edge, of = np.unique(np.sort(t[:, EDGES], -1).reshape(-1, 2), axis=0, return_inverse=True)
    closure = np.concatenate([t, len(p) + of.reshape(-1, 6)], 1)
    nodes = np.concatenate([p, p[edge].mean(1)])
    return mg.Mesh(mg.TET_P2, np.ascontiguousarray(closure, np.int32), np.ascontiguousarray(t, np.int32), p, nodes,
                   None, np.zeros(len(t), np.int32))
