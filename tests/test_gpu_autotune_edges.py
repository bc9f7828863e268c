"""The tuner of batched segments times the walks that intersect_edges and BatchGraph run, and does not take
what was chosen for another kernel."""

import json

import pytest

from tests.test_gpu_subqueries import mesh, queries

pytestmark = pytest.mark.gpu


def test_tunes_what_runs(monkeypatch, tmp_path):
    import numba_celltree_amd as M
    from numba_celltree_amd import batch as B

    trees = [M.CellTree2d(*mesh(k), -1) for k in ("mixed", "triangles")]
    tb = B.TreeBatch(trees)
    segs, counts = B.concat_queries([queries(n, n)[1] for n in (3000, 800)], 4)
    segs = segs.reshape(-1, 2, 2)
    ran = []
    walk = B.gather_edges
    monkeypatch.setattr(B, "gather_edges", lambda plan, *a: ran.append(plan.config) or walk(plan, *a))
    monkeypatch.setattr(B.BatchPlan, "edges_count", lambda *a: pytest.fail("the one-lane count pass"))
    cache = tmp_path / "tuned.json"
    old = ["edges", 2, 3800, tb.max_depth, tb.max_n_vert]
    cache.write_text(json.dumps({json.dumps(old): {"tile": 64, "n_queues": 1, "block": 64}}))
    best, timings = B.autotune(tb, "edges", segs, counts, reps=2, cache_path=str(cache))
    tried = [c for c, _ in timings]
    assert best in tried and len(tried) == len({(c.tile, c.n_queues) for c in tried}) > 4
    assert len(ran) == 3 * len(tried) and set(ran) == set(tried)
    again, timed = B.autotune(tb, "edges", segs, counts, cache_path=str(cache))
    assert again == best and timed == []
