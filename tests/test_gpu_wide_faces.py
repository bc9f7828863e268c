"""Faces of 9 to 24 vertices: the pair stage, the weights and the segment walks of their vertex classes, against
the oracle, with ragged rows (hexagons at the border have fewer sides, and so do their cut forms)."""

import numpy as np
import pytest

from numba_celltree_amd import synthetic as S
from oracle import refcpu as R
from tests.test_gpu_left_over import L, hexagons, queries

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("cuts", [2, 4])
def test_wide_faces_match_oracle(cuts):
    import numba_celltree_amd as M

    v, f = hexagons(cuts)
    g, o = M.CellTree2d(v, f, -1), R.OracleCellTree2d(v, f, -1)
    boxes, seg = queries(600, 40, cuts)
    r = np.random.default_rng(cuts)
    pts = np.concatenate([r.uniform(-1.0, L + 1.0, (3000, 2)), v[::7], 0.5 * (v[f[:200, 0]] + v[f[:200, 1]])])
    print(cuts, "points", flush=True)
    gf, gw = g.compute_barycentric_weights(pts)
    of, ow = o.compute_barycentric_weights(pts)
    assert np.array_equal(gf, of)
    np.testing.assert_allclose(gw, ow, rtol=1e-12, atol=1e-12)
    assert (gw[gf < 0] == 0).all()
    print(cuts, "segments", flush=True)
    for a, b in zip(g.intersect_edges(seg)[:2], o.intersect_edges(seg)[:2]):
        assert np.array_equal(a, b)
    print(cuts, "boxes", flush=True)
    finite = boxes[np.isfinite(boxes).all(axis=1)]
    for a, b in zip(g.intersect_boxes(finite)[:2], o.intersect_boxes(finite)[:2]):
        assert np.array_equal(a, b)
    tv, tf = S.jittered_grid(41, L, 0.25, 0.5, 9)
    for tree, oracle, mesh in ((g, o, (tv, tf)), (M.CellTree2d(tv, tf, -1), R.OracleCellTree2d(tv, tf, -1), (v, f))):
        print(cuts, "faces", len(mesh[1]), flush=True)
        gi, gj, ga = tree.intersect_faces(mesh[0], mesh[1].copy(), -1)
        oi, oj, oa = oracle.intersect_faces(mesh[0], mesh[1].copy(), -1)
        assert np.array_equal(gi, oi) and np.array_equal(gj, oj)
        np.testing.assert_allclose(ga, oa, rtol=1e-12, atol=1e-12 * L * L)
