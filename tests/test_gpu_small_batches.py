"""Point batches small enough to be located by wavefronts that explore a few points' walks at once: the
oracle's first hits, also where several cells hold a point (vertices, edges, stacked cells), for batch
sizes around the points a wavefront takes, leaves of one to many cells, walks with more nodes than lanes
and points that are not finite."""

import numpy as np
import pytest

from numba_celltree_amd import synthetic as S
from oracle import refcpu as R

pytestmark = pytest.mark.gpu


def meshes():
    yield "triangles", *S.jittered_grid(60, 10.0, 0.25, 1.0, 1)
    yield "regular", *S.jittered_grid(41, 10.0, 0.0, 0.5, 1)
    yield "hexagons", *S.hex_voronoi(30, 30, 10.0, 0.1, 2)
    r = np.random.default_rng(5)  # overlapping triangles, many viable leaves and cells for every point
    v = r.uniform(0.0, 10.0, (300, 2))
    yield "stacked", v, np.stack([r.choice(300, 3, replace=False) for _ in range(400)])


@pytest.mark.parametrize("name, v, f", list(meshes()), ids=lambda x: x if isinstance(x, str) else "")
@pytest.mark.parametrize("per_leaf, n_buckets", [(1, 2), (2, 4), (70, 4), (250, 8)])
def test_first_hits(name, v, f, per_leaf, n_buckets):
    import numba_celltree_amd as M

    tree, oracle = M.CellTree2d(v, f, -1, n_buckets, per_leaf), R.OracleCellTree2d(v, f, -1, n_buckets, per_leaf)
    r = np.random.default_rng(per_leaf)
    used = v[np.unique(f[f >= 0])]
    a, b = v[f[:, 0]], v[f[:, 1]]
    pool = np.concatenate([
        used, 0.5 * (a + b), a + r.uniform(0.0, 1.0, (len(f), 1)) * (b - a), r.uniform(-1.0, 11.0, (9000, 2)),
        [[np.nan, 1.0], [1.0, np.nan], [np.inf, 1.0], [-np.inf, np.inf], [0.0, 0.0], [10.0, 10.0]],
    ])
    pool = pool[r.permutation(len(pool))]
    want = oracle.locate_points(pool)
    for n in (1, 2, 15, 16, 17, 4095, 4096, 4097, 8193, len(pool)):
        print(name, per_leaf, n, flush=True)
        assert np.array_equal(tree.locate_points(pool[:n]), want[:n])
    # the largest batch of this kind, one point more, and an order of the points
    many = np.resize(pool, ((1 << 17) + 1, 2))
    got = tree.locate_points(many)
    assert np.array_equal(got, np.resize(want, len(many)))
    assert np.array_equal(tree.locate_points(many[:-1]), got[:-1])

    import torch

    from numba_celltree_amd import _device as D

    d = torch.from_numpy(pool).cuda()
    order = torch.from_numpy(r.permutation(len(pool)).astype(np.int32)).cuda()
    tol = tree._default_tolerance()
    assert np.array_equal(D.Io(pool).out(tree._locate_points_dev(d, tol, order)), want)


@pytest.mark.parametrize("per_leaf", [1, 2, 100])
def test_first_edges(per_leaf):
    import numba_celltree_amd as M

    v, f = S.jittered_grid(40, 10.0, 0.2, 1.0, 1)
    e = np.unique(np.sort(np.concatenate([f[:, [0, 1]], f[:, [1, 2]]]), axis=1), axis=0)
    tree, oracle = M.EdgeCellTree2d(v, e, 4, per_leaf), R.OracleEdgeCellTree2d(v, e, 4, per_leaf)
    r = np.random.default_rng(3)
    p = np.concatenate([v, 0.5 * (v[e[:, 0]] + v[e[:, 1]]), r.uniform(0.0, 10.0, (3000, 2))])
    want = oracle.locate_points(p)
    for n in (1, 16, 17, 4097, len(p)):
        assert np.array_equal(tree.locate_points(p[:n]), want[:n])
