"""Fans of triangles around one vertex: every split cuts a few cells off, so the tree is a chain of
thousands of levels.  Nodes and order are the oracle's, and the time grows with the levels, not with
their square."""

import time

import numpy as np
import pytest

from oracle import refcpu as R

pytestmark = pytest.mark.gpu


def fan(n: int):
    a = np.arange(n) * (2.0 * np.pi / n)
    v = np.concatenate([np.zeros((1, 2)), np.column_stack([np.cos(a), np.sin(a)])])
    i = np.arange(n)
    return v, np.column_stack([np.zeros(n, dtype=np.int64), 1 + i, 1 + (i + 1) % n]).astype(np.int32)


@pytest.mark.parametrize("n", [1500, 4000, 12_000])
def test_chain_of_levels_matches_oracle(n):
    import numba_celltree_amd as M

    v, f = fan(n)
    g, o = M.CellTree2d(v, f, -1), R.OracleCellTree2d(v, f, -1)
    print(n, g.depth, flush=True)
    assert np.array_equal(g.nodes, o.nodes) and np.array_equal(g.bb_indices, o.bb_indices)


def test_time_grows_with_the_levels():
    import torch

    import numba_celltree_amd as M

    def build(n):
        v, f = (torch.from_numpy(a).cuda() for a in fan(n))
        best = float("inf")
        for _ in range(3):
            torch.cuda.synchronize()
            t = time.perf_counter()
            depth = M.CellTree2d(v, f, -1).depth
            torch.cuda.synchronize()
            best = min(best, time.perf_counter() - t)
        print(n, depth, best, flush=True)
        return best

    assert build(80_000) < 10.0 * build(20_000)  # four times the levels
