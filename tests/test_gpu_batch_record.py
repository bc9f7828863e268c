"""Batches with a tree that the wavefront walks do not take are walked by one lane a segment, with a hit
record of many, few and no slots: the rows of every tree's own call, eager and replayed."""

import pytest

from tests.test_gpu_subqueries import mesh, queries

@pytest.mark.gpu
@pytest.mark.parametrize("slots", [256, 8, 0])
def test_batches_with_a_hit_record(monkeypatch, slots):
    import torch

    import numba_celltree_amd as M
    from numba_celltree_amd import batch as B

    trees = [M.CellTree2d(*mesh(k), -1) for k in ("mixed", "hexagons", "triangles")]
    sets = [queries(n, 7 * n)[1] for n in (3000, 1, 800)]
    monkeypatch.setattr(B, "EDGE_HIT_SLOTS", slots)
    tb = B.TreeBatch(trees)
    assert tb.gathers
    want = [t.intersect_edges(torch.from_numpy(s).cuda()) for t, s in zip(trees, sets)]
    for t in trees:
        t.GATHER_MAX_RECORDS = 0
    tb = B.TreeBatch(trees)
    assert not tb.gathers
    segs, counts = B.concat_queries(sets, 4)
    graph = B.BatchGraph(tb, segments=segs.reshape(-1, 2, 2), segment_counts=counts)
    assert graph.buf.slots == slots and graph.buf.pool_rows == 0
    eager = B.intersect_edges(tb, sets)
    for replay in range(3):
        print(slots, replay, flush=True)
        graph.replay()
        res = graph.result()
        for m, w in enumerate(want):
            for rows in (res.edges_of(m), eager[m]):
                assert all(torch.equal(a.view(torch.int64), b.view(torch.int64)) for a, b in zip(rows, w))
