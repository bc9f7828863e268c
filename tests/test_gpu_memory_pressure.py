"""Box and segment batches on a device that holds the row pool but not the rows beside it: the same rows,
without a pool."""

import numpy as np
import pytest

from tests.test_gpu_subqueries import mesh, queries, same

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("long_max", [1 << 20, 0])
def test_rows_without_a_pool(monkeypatch, long_max):
    import torch

    import numba_celltree_amd as M
    from numba_celltree_amd import _device as D

    tree = M.CellTree2d(*mesh("mixed"), -1)
    tree.LONG_MAX = long_max
    boxes, seg = (torch.from_numpy(np.ascontiguousarray(q)).cuda() for q in queries(2000, 4))
    for name, q in (("locate_boxes", boxes), ("intersect_edges", seg)):
        want = [t.cpu().numpy() for t in getattr(tree, name)(q)]
        total = len(want[0])
        failed, held = [], []
        empty = D.empty

        def tight(shape, dtype):
            if shape == total and dtype == torch.int64 and not failed:
                failed.append(torch.cuda.memory_allocated())
                raise torch.cuda.OutOfMemoryError("simulated: no room for the rows")
            if failed and not held:
                held.append(torch.cuda.memory_allocated())
            return empty(shape, dtype)

        monkeypatch.setattr(D, "empty", tight)
        print(long_max, name, total, flush=True)
        same([t.cpu().numpy() for t in getattr(tree, name)(q)], want)
        monkeypatch.setattr(D, "empty", empty)
        assert failed and held[0] < failed[0]  # the first call's pool was given back
