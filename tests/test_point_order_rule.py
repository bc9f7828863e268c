"""Which point batches are located in Morton order: the default rule, and a caller's own ORDERED_MIN."""

import torch

from numba_celltree_amd.celltree import CellTree2d


def tree(cells: int, per_leaf: int) -> CellTree2d:
    t = CellTree2d.__new__(CellTree2d)
    t.d_elements, t.cells_per_leaf = torch.empty((cells, 4), device="meta"), per_leaf
    return t


def test_default_rule():
    small, large = tree(20_000, 2), tree(1_000_000, 2)
    assert not any(small.orders_points(n) for n in (1, 10**6, 10**7))
    assert [large.orders_points(n) for n in (500_000, 10**6, 10**7)] == [False, True, True]
    assert [tree(2000, 16).orders_points(n) for n in (10**6, 1 << 20, 10**7)] == [False, True, True]
    assert [tree(20_000, 64).orders_points(n) for n in (390_000, 400_000)] == [False, True]
    assert [tree(20_000, 130).orders_points(n) for n in (250_000, 270_000)] == [False, True]
    assert not tree(20_000, 7).orders_points(10**7) and tree(20_000, 8).orders_points(10**7)
    assert small.orders_points(1 << 18, vertex_gradients=True)
    assert not small.orders_points((1 << 18) - 1, vertex_gradients=True)


def test_a_callers_value_decides_alone(monkeypatch):
    t = tree(20_000, 2)
    t.ORDERED_MIN = 1000
    assert t.orders_points(1000) and not t.orders_points(999)
    t.ORDERED_MIN = 1 << 18
    assert t.orders_points(1 << 18)
    for t in (tree(20_000, 2), tree(1_000_000, 2), tree(20_000, 500)):
        t.ORDERED_MIN = None
        assert not t.orders_points(10**8) and not t.orders_points(10**8, vertex_gradients=True)
    monkeypatch.setattr(CellTree2d, "ORDERED_MIN", 10)
    assert tree(100, 2).orders_points(10)
