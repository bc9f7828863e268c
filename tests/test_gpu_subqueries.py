"""Trees and batches the wavefront walks do not take (2^26 nodes or cells and more, leaves out of order,
more than 2^29 queries) are cut into subqueries: the rows of the wavefront walks, bit for bit.  The limits
are lowered on the objects here."""

import numpy as np
import pytest

from numba_celltree_amd import synthetic as S

L = 64.0


def test_routes_by_size():
    """The rule alone: nothing is launched, so it runs without a device."""
    import torch

    from numba_celltree_amd import _native
    from numba_celltree_amd.celltree import CellTree2d

    t = CellTree2d.__new__(CellTree2d)
    t.in_order, t.depth, t.n_nodes, t.d_elements = True, 30, 1 << 20, torch.empty((1000, 4), device="meta")
    assert t._gathers(1) and t._gathers(1 << 29)
    assert not t._gathers(0) and not t._splits(0)
    for n in ((1 << 29) + 1, (1 << 31) - 1, 1 << 33):
        assert not t._gathers(n) and t._splits(n)
    t.n_nodes = 1 << 26
    assert not t._gathers(5) and t._splits(5)
    t.n_nodes = 1 << 28
    assert not t._gathers(5) and not t._splits(5)
    t.n_nodes, t.in_order = 1 << 20, False
    assert not t._gathers(5) and t._splits(5)
    t.in_order, t.depth = True, _native.CT_MAX_DEPTH + 1
    assert not t._gathers(5) and not t._splits(5)
    t.depth, t.SPLIT_MAX_PARTS = 30, 1
    assert not t._gathers(5) and not t._splits(5)


def mesh(kind):
    if kind == "hexagons":
        return S.hex_voronoi(40, 40, L, 0.2, 4)
    return S.jittered_grid(61, L, 0.25, 1.0 if kind == "triangles" else 0.5, 4)


def queries(n, seed):
    r = np.random.default_rng(seed)
    c = r.uniform(-3.0, L + 3.0, (n, 2))
    half = 0.5 * np.exp(r.uniform(np.log(0.02), np.log(40.0), (n, 2)))
    boxes = np.column_stack([c[:, 0] - half[:, 0], c[:, 0] + half[:, 0], c[:, 1] - half[:, 1], c[:, 1] + half[:, 1]])
    a, ln = r.uniform(0.0, 2.0 * np.pi, n), np.exp(r.uniform(np.log(0.02), np.log(80.0), n))
    seg = np.stack([c, c + ln[:, None] * np.column_stack([np.cos(a), np.sin(a)])], axis=1)
    seg[::7] = np.round(seg[::7])
    return boxes, seg


def same(got, want):
    for g, w in zip(got, want):
        assert np.array_equal(g.view(np.int64), w.view(np.int64))


@pytest.mark.gpu
@pytest.mark.parametrize("kind", ["mixed", "hexagons", "edges"])
@pytest.mark.parametrize("n, max_parts, leaf_cells, slots", [(1, 16, 32, 64), (900, 2, 2, 4), (5000, 7, 4, 0),
                                                             (5000, 16, 1, 64), (5000, 16, 16, 1024)])
def test_subqueries_have_the_rows_of_wavefront_walks(monkeypatch, kind, n, max_parts, leaf_cells, slots):
    import numba_celltree_amd as M

    v, f = mesh(kind)
    if kind == "edges":
        fv = f[:, :3]
        tree = M.EdgeCellTree2d(v, np.unique(np.sort(np.concatenate([fv[:, :2], fv[:, 1:]]), axis=1), axis=0))
    else:
        tree = M.CellTree2d(v, f, -1)
    boxes, seg = queries(n, 3 * n + slots)
    calls = [("intersect_edges", seg)] + ([] if kind == "edges" else [("locate_boxes", boxes)])
    want = [getattr(tree, name)(q) for name, q in calls]
    ran = []
    split = type(tree)._split_rows
    monkeypatch.setattr(type(tree), "_split_rows", lambda self, *a: ran.append(a[0]) or split(self, *a))
    tree.GATHER_MAX_RECORDS = 0
    tree.SPLIT_MIN_CELLS, tree.SPLIT_MAX_PARTS = 0, max_parts
    tree.SPLIT_LEAF_CELLS = tree.EDGE_SPLIT_LEAF_CELLS = leaf_cells
    tree.BOX_HIT_SLOTS = tree.EDGE_HIT_SLOTS = max(slots, 1)
    tree.BOX_HIT_BUDGET = tree.EDGE_HIT_BUDGET = slots * 10**6
    tree.EDGE_XY_SLOTS = {4: 4, 0: 0, 64: 16, 1024: 1024}[slots]
    for (name, q), w in zip(calls, want):
        print(kind, n, slots, name, flush=True)
        same(getattr(tree, name)(q), w)
    assert len(ran) == len(calls)

