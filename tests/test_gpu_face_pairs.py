"""intersect_faces settles most separating-axis tests by a point well inside both faces: the pairs it
keeps and their areas have to be those of the test itself (polygons_intersect) and of the clip
(area_of_intersection) run on their own, bit for bit, and the oracle's pairs: faces that touch, that
overlap by next to nothing, far from and around the origin, very small and very large, not convex,
self-intersecting and degenerate."""

import numpy as np
import pytest

from numba_celltree_amd import synthetic as S
from oracle import refcpu as R

pytestmark = pytest.mark.gpu


def quads(n: int, length: float):
    x = np.linspace(0.0, length, n + 1)
    v = np.stack(np.meshgrid(x, x), axis=-1).reshape(-1, 2)
    k = (np.arange(n)[:, None] * (n + 1) + np.arange(n)[None, :]).reshape(-1)
    return v, np.stack([k, k + 1, k + n + 2, k + n + 1], axis=1)


def odd(width: int, n: int, seed: int):
    """Random rows of 3..width vertices of a small cloud: not convex, crossing, with repeated vertices."""
    r = np.random.default_rng(seed)
    v = np.round(r.uniform(0.0, 4.0, (60, 2)) * 8.0) / 8.0
    f = np.full((n, width), -1, dtype=np.int64)
    for i in range(n):
        k = int(r.integers(3, width + 1))
        f[i, :k] = r.choice(60, k, replace=i % 5 == 0)
    return v, f


def cases():
    yield "same quads", quads(12, 4.0), quads(12, 4.0)
    yield "aligned", quads(12, 4.0), quads(9, 3.0)
    for e in (1e-3, 1e-7, 1e-9, 1e-11, 1e-12, 1e-13, 1e-15):
        v, f = quads(12, 4.0)
        yield f"shifted {e}", quads(12, 4.0), (v + np.array([e, -0.7 * e]), f)
        v, f = S.jittered_grid(13, 4.0, 0.2, 0.5, 1)
        yield f"jittered {e}", (v, f), (v * (1.0 + e) + e, f)
    grid, hexagons = S.jittered_grid(13, 4.0, 0.2, 0.5, 1), S.hex_voronoi(8, 8, 4.0, 0.1, 2)
    for name, move, scale in (("origin", -2.0, 1.0), ("far", 3e5, 1.0), ("tiny", 0.0, 1e-90), ("tinier", 0.0, 1e-153),
                              ("large", 0.0, 1e90)):
        yield name, *(((v + move) * scale, f) for v, f in (grid, hexagons))
        yield name + " back", *(((v + move) * scale, f) for v, f in (hexagons, grid))
    for width in (3, 4, 6, 12):
        yield f"odd {width}", odd(width, 80, width), odd(width, 90, 100 + width)
        yield f"odd onto grid {width}", grid, odd(width, 90, 200 + width)


@pytest.mark.parametrize("name, src, tgt", list(cases()), ids=lambda x: x if isinstance(x, str) else "")
def test_pairs_and_areas(name, src, tgt):
    import torch

    import numba_celltree_amd as M
    from numba_celltree_amd import algorithms as A

    tree = M.CellTree2d(src[0], src[1], -1)
    tv, tf = torch.from_numpy(tgt[0]).cuda(), torch.from_numpy(tgt[1]).cuda()
    d_v, d_f, prep = tree._faces_in(tv, tf, -1)
    bb = tree._prepare_faces(d_v, d_f) if prep is None else prep.bb
    ii, jj = tree._locate_boxes_dev(bb, prep)
    sat = A.polygons_intersect(d_v, tree.d_vertices, d_f, tree.d_elements, ii, jj).bool()
    area = A.area_of_intersection(d_v, tree.d_vertices, d_f, tree.d_elements, ii, jj)
    keep = sat & (area > 0)
    gi, gj, ga = tree.intersect_faces(tv, tf, -1)
    assert torch.equal(gi, ii[keep]) and torch.equal(gj, jj[keep])
    assert torch.equal(ga.view(torch.int64), area[keep].view(torch.int64))
    # the int64 flags of the C entry
    from numba_celltree_amd import _device as D
    from numba_celltree_amd import _native

    n = int(ii.numel())
    a2, k2 = D.empty(n, torch.float64), D.empty(n, torch.int64)
    _native.call("ct_face_pairs", D.ptr(d_v), D.ptr(d_f), int(d_f.shape[1]), D.ptr(tree.d_vertices),
                 D.ptr(tree.d_elements), int(tree.d_elements.shape[1]), D.ptr(ii), D.ptr(jj), n, 1, D.ptr(a2),
                 D.ptr(k2), D.stream())
    assert torch.equal(k2.bool(), keep)
    assert torch.equal(a2, torch.where(sat, area, torch.zeros_like(area)))
    oi, oj, _ = R.OracleCellTree2d(src[0], src[1], -1).intersect_faces(tgt[0], tgt[1].copy(), -1)
    assert np.array_equal(gi.cpu().numpy(), oi) and np.array_equal(gj.cpu().numpy(), oj)
