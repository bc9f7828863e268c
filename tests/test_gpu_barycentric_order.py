"""Vertex gradients of the barycentric adjoints with the points in Morton order (a face's points are
summed in a wavefront before they are added) and without: both against the sum of every point's own
contributions, taken one by one from a mesh in which no two points share a vertex."""

import numpy as np
import pytest

from numba_celltree_amd import synthetic as S

pytestmark = pytest.mark.gpu


def _gradients(points, vertices, faces, face, tol, wachspress, order, G):
    import torch

    from numba_celltree_amd.barycentric import BarycentricFunction

    p, v = points.clone().requires_grad_(), vertices.clone().requires_grad_()
    w = BarycentricFunction.apply(p, v, faces, face, tol, wachspress, order)
    return torch.autograd.grad(w, (p, v), G)


@pytest.mark.parametrize("kind", ["triangles", "mixed", "hexagons", "wide"])
@pytest.mark.parametrize("n", [1, 3, 64, 65, 257, 20_000])
def test_ordered_sums(kind, n):
    import torch

    import numba_celltree_amd as M
    from numba_celltree_amd import _device as D

    if kind in ("hexagons", "wide"):
        v, f = S.hex_voronoi(8, 8, 10.0, 0.1, 5)
        if kind == "wide":
            f = np.concatenate([f, np.full((len(f), 12 - f.shape[1]), -1, f.dtype)], axis=1)
    else:
        v, f = S.jittered_grid(12, 10.0, 0.2, 1.0 if kind == "triangles" else 0.4, 2)
    tree = M.CellTree2d(v, f, -1)
    rng = np.random.default_rng(n)
    pts = torch.from_numpy(rng.uniform(-0.5, 10.5, (n, 2))).cuda()
    pts[n // 2:] = pts[n // 2:] * 0.05 + 4.0  # half of them crowd into a few faces
    faces, wachspress = tree.d_elements, int(tree.d_elements.shape[1]) > 3
    k = int(faces.shape[1]) if wachspress else 3
    tol = tree._default_tolerance()
    face = tree._locate_points_dev(pts, tol)
    G = torch.from_numpy(rng.normal(size=(n, k))).cuda()
    # every point its own copy of its face
    cols = int(faces.shape[1])
    rows = faces[face.clamp(min=0)]
    own = torch.arange(n * cols, device="cuda").reshape(n, cols)
    own_faces = torch.where(rows < 0, -1, own).to(torch.int32).contiguous()
    own_vertices = tree.d_vertices[rows.clamp(min=0).long()].reshape(-1, 2).contiguous()
    own_face = torch.where(face < 0, -1, torch.arange(n, device="cuda"))
    gp, each = _gradients(pts, own_vertices, own_faces, own_face, tol, wachspress, None, G)
    at = rows.clamp(min=0).long().reshape(-1).cpu()
    each = each.cpu()
    each[(rows < 0).reshape(-1).cpu()] = 0.0
    want = torch.zeros(len(v), 2, dtype=torch.float64).index_add_(0, at, each)
    size = torch.zeros(len(v), 2, dtype=torch.float64).index_add_(0, at, each.abs())
    terms = torch.zeros(len(v), dtype=torch.float64).index_add_(0, at, torch.ones(len(at), dtype=torch.float64))
    bound = 2.0 * terms[:, None] * np.finfo(np.float64).eps * size  # of two sums in any order
    for order in (None, D.query_order(0, pts, tree._bbox)):
        gp2, gv = _gradients(pts, tree.d_vertices, faces, face, tol, wachspress, order, G)
        assert torch.equal(gp2, gp)
        assert bool(((gv.cpu() - want).abs() <= bound).all())
