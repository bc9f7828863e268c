"""Queries that a wavefront walk leaves over, merged with those it keeps: walked by a wavefront each
(ct_long_*) or as subqueries, with the rows of whole walks bit for bit and in the same order, and the
oracle's.  Left for their rows (more than the lists hold) or for the pool (budgets of some rows, fewer than
the batch has); faces of every vertex class and edges."""

import numpy as np
import pytest

from numba_celltree_amd import synthetic as S
from oracle import refcpu as R

pytestmark = pytest.mark.gpu

L = 64.0


def hexagons(cuts: int):
    """A honeycomb whose sides are cut into `cuts` pieces each: faces of up to 6 * cuts vertices."""
    v, f = S.hex_voronoi(36, 36, L, 0.2, 4)
    pts, faces = [], []
    for row in f:
        p = v[row[row >= 0]]
        q = np.roll(p, -1, axis=0)
        ring = np.concatenate([p + (q - p) * (k / cuts) for k in range(cuts)], axis=1).reshape(-1, 2)
        faces.append(np.arange(len(ring)) + sum(map(len, pts)))
        pts.append(ring)
    out = np.full((len(faces), max(map(len, faces))), -1, dtype=np.int32)
    for i, row in enumerate(faces):
        out[i, : len(row)] = row
    return np.concatenate(pts), out


def trees(kind):
    import numba_celltree_amd as M

    if kind == "edges":
        v, f = S.jittered_grid(201, L, 0.25, 1.0, 4)
        e = np.unique(np.sort(np.concatenate([f[:, [0, 1]], f[:, [1, 2]]]), axis=1), axis=0)
        return M.EdgeCellTree2d(v, e), R.OracleEdgeCellTree2d(v, e), None
    if kind.startswith("hexagons"):
        v, f = hexagons(int(kind[-1]))
        if kind == "hexagons1":
            v, f = S.hex_voronoi(130, 130, L, 0.2, 4)
    else:
        v, f = S.jittered_grid(181, L, 0.25, 0.5, 4)
    per_leaf = 300 if kind == "leaves" else 2
    return M.CellTree2d(v, f, -1, 4, per_leaf), R.OracleCellTree2d(v, f, -1, 4, per_leaf), f


def queries(n, big, seed):
    """n small boxes and segments, every `big`-th large: up to the whole square."""
    r = np.random.default_rng(seed)
    c = r.uniform(-2.0, L + 2.0, (n, 2))
    half = 0.5 * np.exp(r.uniform(np.log(0.02), np.log(4.0), (n, 2)))
    a, ln = r.uniform(0.0, 2.0 * np.pi, n), np.exp(r.uniform(np.log(0.02), np.log(8.0), n))
    half[::big] = r.uniform(0.2 * L, 0.7 * L, (len(half[::big]), 2))
    c[::big] = r.uniform(0.0, 0.3 * L, c[::big].shape)
    ln[::big] = r.uniform(0.7 * L, 1.3 * L, len(ln[::big]))
    a[::big] = r.uniform(0.0, 0.5 * np.pi, len(a[::big]))
    boxes = np.column_stack([c[:, 0] - half[:, 0], c[:, 0] + half[:, 0], c[:, 1] - half[:, 1], c[:, 1] + half[:, 1]])
    seg = np.stack([c, c + ln[:, None] * np.column_stack([np.cos(a), np.sin(a)])], axis=1)
    seg[::7] = np.round(seg[::7])  # along mesh lines and through vertices: ties in t
    seg[5], boxes[5] = [[np.nan, 1.0], [2.0, 3.0]], [1.0, np.inf, 2.0, np.nan]
    seg[6], boxes[6] = [[1.0, 1.0], [np.inf, 3.0]], [-np.inf, np.inf, -np.inf, np.inf]
    return boxes, seg


def spy(monkeypatch, cls):
    """The numbers of queries left to _count_long and to _count_subs."""
    seen = {"long": [], "subs": []}
    count_long, count_subs = cls._count_long, cls._count_subs
    monkeypatch.setattr(cls, "_count_long", lambda self, k, q, ids, m, *a: seen["long"].append(m)
                        or count_long(self, k, q, ids, m, *a))
    monkeypatch.setattr(cls, "_count_subs", lambda self, k, q, o, m, *a: seen["subs"].append(m)
                        or count_subs(self, k, q, o, m, *a))
    return seen


def check(tree, oracle, name, q):
    got = getattr(tree, name)(q)
    tree.SPLIT_MAX_PARTS = 1  # whole walks
    want = getattr(tree, name)(q)
    del tree.SPLIT_MAX_PARTS
    for g, w in zip(got, want):
        assert np.array_equal(g.view(np.int64), w.view(np.int64))
    ref = getattr(oracle, name)(q)
    assert np.array_equal(got[0], ref[0]) and np.array_equal(got[1], ref[1])
    return len(got[0])


@pytest.mark.parametrize("kind", ["mixed", "leaves", "hexagons1", "hexagons2", "hexagons4", "edges"])
@pytest.mark.parametrize("n", [40, 3000])
@pytest.mark.parametrize("by", ["wavefronts", "subqueries"])
def test_large_queries_among_small_ones(monkeypatch, kind, n, by):
    tree, oracle, _ = trees(kind)
    seen = spy(monkeypatch, type(tree))
    if by == "subqueries":
        tree.LONG_MAX = 0
    boxes, seg = queries(n, 10, n)
    for name, q in [("intersect_edges", seg)] + ([] if kind == "edges" else [("locate_boxes", boxes)]):
        print(kind, n, by, name, flush=True)
        for k in seen:
            seen[k].clear()
        check(tree, oracle, name, q)
        left = seen["long" if by == "wavefronts" else "subs"]
        if not (kind in ("hexagons2", "hexagons4") and name == "intersect_edges"):  # 36 cells across
            assert left and 0 < left[0] < n / 2, seen


@pytest.mark.parametrize("kind", ["mixed", "hexagons1", "edges"])
@pytest.mark.parametrize("by", ["wavefronts", "subqueries"])
def test_pools_that_run_out(monkeypatch, kind, by):
    """Budgets that hold some of a batch's rows: kept queries beside left ones, and boxes that the pool takes
    on their second walk beside those it does not."""
    tree, oracle, _ = trees(kind)
    seen = spy(monkeypatch, type(tree))
    if by == "subqueries":
        tree.LONG_MAX = 0
    boxes, seg = queries(3000, 10**9, 3)
    for name, q in [("intersect_edges", seg)] + ([] if kind == "edges" else [("locate_boxes", boxes)]):
        for k in seen:
            seen[k].clear()
        rows = check(tree, oracle, name, q)
        assert sum(seen["long"] + seen["subs"]) <= 3  # the first, large, and the infinite ones
        kept = []
        for share in (1.2, 0.9, 0.6, 0.3, 0.1, 0.0):
            for k in seen:
                seen[k].clear()
            print(kind, by, name, share, flush=True)
            tree.BOX_HIT_BUDGET = int(share * rows)
            tree.EDGE_HIT_BUDGET = int(share * 2 * (1.5 * rows + 34 * 3000))  # two words a row, what groups ask for
            check(tree, oracle, name, q)
            left = seen["long" if by == "wavefronts" else "subs"]
            kept.append(3000 - left[0] if left else 3000)
        del tree.BOX_HIT_BUDGET, tree.EDGE_HIT_BUDGET
        print(kept, flush=True)
        assert kept == sorted(kept, reverse=True)
        assert any(1500 < k < 3000 for k in kept) and any(0 < k < 1500 for k in kept), kept


@pytest.mark.parametrize("n", [300, 20_000])
def test_equal_queries_up_to_the_lists_are_kept(monkeypatch, n):
    """Boxes of up to 20 and segments of up to 130 cell sides, all alike: the pool has room for every one."""
    import torch

    import numba_celltree_amd as M

    v, f = S.jittered_grid(301, L, 0.25, 1.0 / 3.0, 4)
    tree = M.CellTree2d(v, f, -1)
    seen = spy(monkeypatch, type(tree))
    h, r = L / 300, np.random.default_rng(n)
    c, a = r.uniform(0.0, L, (n, 2)), r.uniform(0.0, 2.0 * np.pi, n)
    for side in (5, 14, 20):
        w = 0.5 * side * h
        b = np.column_stack([c[:, 0] - w, c[:, 0] + w, c[:, 1] - w, c[:, 1] + w])
        print(n, side, len(tree.locate_boxes(torch.from_numpy(b).cuda())[0]), flush=True)
    for side in (20, 70, 130):
        d = side * h * np.column_stack([np.cos(a), np.sin(a)])
        print(n, side, len(tree.intersect_edges(torch.from_numpy(np.stack([c, c + d], axis=1)).cuda())[0]), flush=True)
    assert not seen["long"] and not seen["subs"]


def test_few_boxes_over_all_cells_are_walked_once(monkeypatch):
    """Boxes whose expected number of rows is more than the mesh has cells, one and several."""
    from numba_celltree_amd import _native

    tree, oracle, f = trees("mixed")
    written = []
    call = _native.call
    monkeypatch.setattr(_native, "call", lambda name, *a: written.append(name) or call(name, *a))
    for n in (1, 7):
        boxes = np.tile([[-3.0 * L, 4.0 * L, -1.0, L + 1.0]], (n, 1))
        ii, jj = tree.locate_boxes(boxes)
        oi, oj = oracle.locate_boxes(boxes)
        assert np.array_equal(ii, oi) and np.array_equal(jj, oj) and len(ii) == n * len(f)
    assert "ct_long_count" in written
    # every box is in the pool after its first walk
    import torch

    starts = []
    long_boxes = type(tree)._count_long

    def keep(self, k, q, ids, m, rows, cell, counts, st, tail):
        starts.append(st)
        return long_boxes(self, k, q, ids, m, rows, cell, counts, st, tail)

    monkeypatch.setattr(type(tree), "_count_long", keep)
    tree.locate_boxes(torch.from_numpy(boxes).cuda())
    assert bool((starts[0] >= 0).all())


def test_pool_stays_within_the_budgets():
    """Two int32 and 32 bytes of a piece per row, whatever the batch asks for."""
    import torch

    tree, oracle, _ = trees("mixed")
    _, seg = queries(3000, 10, 1)
    asked = []
    pool = type(tree)._pool

    def record(rows, widths):
        asked.append(rows)
        return pool(rows, widths)

    tree._pool = record
    for hit, xy in ((1 << 28, 1 << 32), (5000, 1 << 32), (1 << 28, 3200)):
        tree.EDGE_HIT_BUDGET, tree.EDGE_XY_BUDGET = hit, xy
        tree.intersect_edges(torch.from_numpy(seg).cuda())
        assert asked[-1] <= min(hit // 2, xy // 32)
