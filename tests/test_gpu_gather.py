"""Box and segment queries walked by wavefronts (ct_gather_*) have the rows of the whole walks, bit for
bit and in the same order, and the oracle's: queries per wavefront from 1 to 16, leaves from one cell to
more than a wavefront lists, rows per query from none to more than its lists hold (left to the
subqueries), ties in t, segments that are not finite, and pools that run out."""

import numpy as np
import pytest

from numba_celltree_amd import synthetic as S
from oracle import refcpu as R

pytestmark = pytest.mark.gpu

L = 64.0


def mesh(kind: str):
    if kind == "hexagons":
        return S.hex_voronoi(60, 60, L, 0.2, 4)
    jitter = 0.0 if kind == "ties" else 0.25
    return S.jittered_grid(65, L, jitter, 0.5, 4)


def queries(n: int, seed: int):
    r = np.random.default_rng(seed)
    c = r.uniform(-3.0, L + 3.0, (n, 2))
    half = 0.5 * np.exp(r.uniform(np.log(0.02), np.log(4.0 if n > 5000 else 60.0), (n, 2)))
    boxes = np.column_stack([c[:, 0] - half[:, 0], c[:, 0] + half[:, 0], c[:, 1] - half[:, 1], c[:, 1] + half[:, 1]])
    a = r.uniform(0.0, 2.0 * np.pi, n)
    length = np.exp(r.uniform(np.log(0.02), np.log(8.0 if n > 5000 else 90.0), n))
    d = length[:, None] * np.column_stack([np.cos(a), np.sin(a)])
    seg = np.stack([c, c + d], axis=1)
    seg[::7] = np.round(seg[::7])  # along mesh lines and through vertices
    seg[3::11, 1, 1] = seg[3::11, 0, 1]
    if n > 60:
        boxes[5] = [-1.0, L + 1.0, -1.0, L + 1.0]
        seg[5] = [[-1.0, -1.0], [L + 1.0, L + 1.0]]
        seg[17, 1, 0], seg[29, 0, 1], seg[41, 1] = np.nan, np.inf, [-np.inf, np.inf]
        boxes[23, 1], boxes[47, 2] = np.inf, np.nan
    return boxes, seg


@pytest.mark.parametrize("kind, per_leaf", [("mixed", 2), ("ties", 1), ("hexagons", 3), ("mixed", 40), ("ties", 250),
                                            ("edges", 2)])
@pytest.mark.parametrize("n, budget", [(1, None), (63, None), (5000, None), (5000, 3000), (5000, 0), (70000, None)])
def test_rows_of_whole_walks(kind, per_leaf, n, budget):
    import numba_celltree_amd as M

    v, f = mesh(kind)
    if kind == "edges":
        fv = f[:, :3]
        e = np.unique(np.sort(np.concatenate([fv[:, [0, 1]], fv[:, [1, 2]]]), axis=1), axis=0)
        tree, oracle = M.EdgeCellTree2d(v, e, 4, per_leaf), R.OracleEdgeCellTree2d(v, e, 4, per_leaf)
    else:
        tree, oracle = M.CellTree2d(v, f, -1, 4, per_leaf), R.OracleCellTree2d(v, f, -1, 4, per_leaf)
    if n > 5000:
        tree.GATHER_ORDER_MIN = tree.GATHER_ORDER_CELLS = 0
    boxes, seg = queries(n, 7 * n + per_leaf)
    calls = [("intersect_edges", seg)] + ([] if kind == "edges" else [("locate_boxes", boxes)])
    for name, q in calls:
        print(kind, per_leaf, n, budget, name, flush=True)
        if budget is not None:
            tree.BOX_HIT_BUDGET = tree.EDGE_HIT_BUDGET = budget
        got = getattr(tree, name)(q)
        tree.SPLIT_MAX_PARTS = 1  # whole walks
        want = getattr(tree, name)(q)
        del tree.SPLIT_MAX_PARTS
        for g, w in zip(got, want):
            assert np.array_equal(g, w, equal_nan=g.dtype.kind == "f")
        ref = getattr(oracle, name)(q)
        assert np.array_equal(got[0], ref[0]) and np.array_equal(got[1], ref[1])


@pytest.mark.parametrize("tile, slots", [(64, 256), (1024, 256), (256, 8), (256, 0)])
def test_batched_rows_of_single_calls(monkeypatch, tile, slots):
    """A captured batch of segments, some of more rows than a wavefront's lists hold, and pools that
    suffice, run out or are absent: the rows of every tree's own call, on every replay."""
    import torch

    import numba_celltree_amd as M
    from numba_celltree_amd import batch as B

    monkeypatch.setattr(B, "EDGE_HIT_SLOTS", slots)
    meshes = [mesh("mixed"), S.jittered_grid(200, L, 0.2, 0.5, 9), mesh("hexagons"), mesh("ties")]
    trees = [M.CellTree2d(torch.from_numpy(v).cuda(), torch.from_numpy(f).cuda(), -1) for v, f in meshes]
    sets = [queries(n, 11 * n)[1] for n in (1, 700, 5000, 130)]
    sets[1][5] = [[-1.0, -1.0], [L + 1.0, L + 0.5]]  # crosses some 600 cells
    tb = B.TreeBatch(trees)
    segs, counts = B.concat_queries(sets, 4)
    graph = B.BatchGraph(tb, segments=segs.reshape(-1, 2, 2), segment_counts=counts,
                         edges_config=B.BatchConfig(tile=tile))
    want = [t.intersect_edges(torch.from_numpy(s).cuda()) for t, s in zip(trees, sets)]
    assert max(int(torch.bincount(w[0]).max()) for w in want) > 320
    for replay in range(3):
        print(tile, slots, replay, flush=True)
        graph.buf.jj_sorted.fill_(-7)
        graph.replay()
        res = graph.result()
        for m, w in enumerate(want):
            got = res.edges_of(m)
            assert torch.equal(got[0], w[0]) and torch.equal(got[1], w[1])
            assert torch.equal(got[2].view(torch.int64), w[2].view(torch.int64))
