"""Imported trees whose leaves do not lie in tree order: accepted (ct_check_tree bounds their ranges
only), told apart (ct_leaves_in_order), and answered as the oracle walks them."""

import numpy as np
import pytest

from numba_celltree_amd import synthetic as S
from numba_celltree_amd import treeio
from oracle import refcpu as R

L = 100.0


def tree_with(leaves: str, per_leaf: int = 3):
    """An oracle tree whose leaves lie as built, in the opposite order, or beginning one position early
    (and so overlapping the leaf before)."""
    v, f = S.jittered_grid(41, L, 0.25, 1.0 / 3.0, 6)
    o = R.OracleCellTree2d(v, f, -1, 4, per_leaf)
    leaf = np.flatnonzero(o.nodes["child"] == -1)
    if leaves == "reversed":
        order = leaf[np.argsort(-o.nodes["ptr"][leaf])]
        cells = [o.bb_indices[o.nodes["ptr"][i]: o.nodes["ptr"][i] + o.nodes["size"][i]].copy() for i in order]
        o.nodes["ptr"][order] = np.concatenate([[0], np.cumsum(o.nodes["size"][order])[:-1]])
        o.bb_indices[:] = np.concatenate(cells)
    elif leaves == "overlapping":
        grow = leaf[(o.nodes["ptr"][leaf] > 0) & (np.arange(len(leaf)) % 3 == 0)]
        o.nodes["ptr"][grow] -= 1
        o.nodes["size"][grow] += 1
    return o


def arrays(o):
    return {"vertices": o.vertices, "elements": o.faces, "nodes": o.nodes, "bb_indices": o.bb_indices,
            "n_buckets": 4, "cells_per_leaf": 3, "kind": "faces"}


def test_leaves_in_order_of_small_trees():
    assert treeio.validate(arrays(tree_with("built")))["in_order"]
    for leaves in ("reversed", "overlapping"):
        assert not treeio.validate(arrays(tree_with(leaves)))["in_order"], leaves
    one = np.zeros(1, dtype=treeio.NODE_RECORD)
    one["child"], one["size"] = -1, 5
    assert treeio.leaves_in_order(one, 5) and not treeio.leaves_in_order(one, 6)
    three = np.zeros(3, dtype=treeio.NODE_RECORD)
    three["child"], three["size"], three["ptr"] = [1, -1, -1], [7, 3, 4], [0, 0, 3]
    assert treeio.leaves_in_order(three, 7)
    three["ptr"][1:] = [4, 0]  # the right leaf first
    assert not treeio.leaves_in_order(three, 7)


@pytest.mark.gpu
@pytest.mark.parametrize("leaves", ["built", "reversed", "overlapping"])
def test_imported_leaf_orders_match_oracle(leaves):
    import torch

    import numba_celltree_amd as M
    from numba_celltree_amd import batch as B

    o = tree_with(leaves)
    g = M.CellTree2d.from_arrays(**arrays(o))
    assert g.in_order == (leaves == "built")
    r = np.random.default_rng(8)
    c, w = r.uniform(-5.0, L + 5.0, (3000, 2)), np.exp(r.uniform(np.log(0.1), np.log(30.0), (3000, 2)))
    boxes = np.column_stack([c[:, 0] - w[:, 0], c[:, 0] + w[:, 0], c[:, 1] - w[:, 1], c[:, 1] + w[:, 1]])
    seg = np.stack([c, r.uniform(-5.0, L + 5.0, (3000, 2))], axis=1)
    seg[::5] = np.round(seg[::5])
    for name, q in (("locate_boxes", boxes), ("intersect_edges", seg), ("locate_points", c)):
        print(leaves, name, flush=True)
        got, want = getattr(g, name)(q), getattr(o, name)(q)
        for a, b in zip(np.atleast_2d(got)[:2] if name == "locate_points" else got[:2],
                        np.atleast_2d(want)[:2] if name == "locate_points" else want[:2]):
            assert np.array_equal(a, b), name
    print(leaves, "batch", flush=True)
    tb = B.TreeBatch([g, g])
    rows = B.intersect_edges(tb, [torch.from_numpy(seg[:1000]).cuda(), torch.from_numpy(seg[1000:]).cuda()])
    for (gi, gj, _), part in zip(rows, (seg[:1000], seg[1000:])):
        oi, oj, _ = o.intersect_edges(part)
        assert np.array_equal(gi.cpu().numpy(), oi) and np.array_equal(gj.cpu().numpy(), oj)
