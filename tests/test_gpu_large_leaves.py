"""Wavefront walks of trees with leaves around and past the cells a wavefront lists at once: no query is
left over for its leaves, and the rows are the oracle's."""

import numpy as np
import pytest

from numba_celltree_amd import synthetic as S
from oracle import refcpu as R
from tests.test_gpu_subqueries import L, queries

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("per_leaf", [63, 64, 65, 128, 192, 193, 400, 5000])
def test_no_query_is_left_for_its_leaves(per_leaf):
    import torch

    import numba_celltree_amd as M
    from numba_celltree_amd import _device as D
    from numba_celltree_amd import _native

    v, f = S.jittered_grid(61, L, 0.25, 1.0, 4)
    tree, oracle = M.CellTree2d(v, f, -1, 4, per_leaf), R.OracleCellTree2d(v, f, -1, 4, per_leaf)
    boxes, seg = queries(400, per_leaf)
    c = 0.5 * (boxes[:, 0::2] + boxes[:, 1::2])
    boxes = np.column_stack([c[:, 0] - 2.0, c[:, 0] + 2.0, c[:, 1] - 2.0, c[:, 1] + 2.0])
    seg = seg[np.hypot(*(seg[:, 1] - seg[:, 0]).T) < 20.0]
    for kind, q, name in ((1, boxes, "locate_boxes"), (2, seg, "intersect_edges")):
        print(per_leaf, name, flush=True)
        d, n = torch.from_numpy(np.ascontiguousarray(q)).cuda(), len(q)
        rows = 1 << 20
        pool = [D.empty(rows, torch.int32), D.empty((rows, 4), torch.float64), D.empty(rows, torch.int32)]
        counts, starts = D.empty(n, torch.int64), D.empty(n, torch.int64)
        tail = D.empty(int(_native.lib().ct_gather_tail_words()), torch.int64)
        _native.call("ct_gather_count", tree.tree_ref, kind, D.ptr(d), n, 0, D.ptr(tree.d_visit_cells), rows,
                     *(D.ptr(t) for t in pool), D.ptr(counts), D.ptr(starts), D.ptr(tail), D.stream())
        assert int(tail[0]) == 0 and bool((starts >= 0).all())
        got, want = getattr(tree, name)(q), getattr(oracle, name)(q)
        assert np.array_equal(got[0], want[0]) and np.array_equal(got[1], want[1])
