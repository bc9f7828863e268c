"""Device face arrays take one fused pass (conversion, index checks, counter-clockwise order, boxes);
host arrays take the separate ones.  Both have to give the same tree and the same overlaps, and
raise the same errors, for every width, index type, fill value and row order."""

import numpy as np
import pytest

from numba_celltree_amd import synthetic as S

pytestmark = pytest.mark.gpu

N_VERTICES = 400


def polygons(width: int, n: int, seed: int):
    """Convex and degenerate rows of 3..width vertices, half of them clockwise, -1 padded."""
    r = np.random.default_rng([seed, width])
    v = r.uniform(0.0, 10.0, (N_VERTICES, 2))
    f = np.full((n, width), -1, dtype=np.int64)
    for i in range(n):
        k = int(r.integers(3, width + 1))
        row = r.choice(N_VERTICES, k, replace=False)
        c = v[row].mean(0)
        row = row[np.argsort(np.arctan2(v[row, 1] - c[1], v[row, 0] - c[0]))]
        if i % 2:
            row = row[::-1]
        if i % 11 == 0:
            row[1] = row[0]  # a repeated vertex
        f[i, :k] = row
    v[7] = v[8]
    return v, f


@pytest.mark.parametrize("width", [3, 4, 5, 8])
@pytest.mark.parametrize("dtype,fill", [(np.int32, -1), (np.int64, -1), (np.int64, -999), (np.int32, 99999)])
@pytest.mark.parametrize("n", [1, 255, 257, 3000])
def test_same_tree_as_host_arrays(width, dtype, fill, n):
    import torch

    import numba_celltree_amd as M

    v, f = polygons(width, n, 3)
    f = np.where(f == -1, fill, f).astype(dtype)
    host = M.CellTree2d(v, f, fill)
    dev = M.CellTree2d(torch.from_numpy(v).cuda(), torch.from_numpy(f).cuda(), fill)
    for name in ("d_elements", "d_bb_coords", "d_nodes", "d_bb_indices", "d_bb_distances"):
        assert torch.equal(getattr(host, name), getattr(dev, name)), name
    assert np.array_equal(host.bbox, dev.bbox) and host._max_diagonal == dev._max_diagonal


@pytest.mark.parametrize("n", [3, 5000])
def test_same_overlaps_as_host_arrays(n):
    import torch

    import numba_celltree_amd as M

    v, f = S.jittered_grid(41, 10.0, 0.2, 0.5, 1)
    tree = M.CellTree2d(v, f, -1)
    tv, tf = S.jittered_grid(72, 10.0, 0.2, 0.3, 2)
    tf = tf[:n]
    want = tree.intersect_faces(tv, np.where(tf == -1, -9, tf), -9)
    d_tf = torch.from_numpy(tf).cuda()
    # a strided view, int64 with another fill value
    wide = torch.stack([torch.where(d_tf == -1, -9, d_tf).long()] * 2, dim=2)
    got = tree.intersect_faces(torch.from_numpy(tv).cuda(), wide[:, :, 0], -9)
    for a, b in zip(want, got):
        assert np.array_equal(a, b.cpu().numpy())
    assert torch.equal(d_tf.cpu(), torch.from_numpy(tf))  # the caller's rows stay as they are


@pytest.mark.parametrize("bad,match", [(N_VERTICES, "out of bounds"), (2**40, "out of bounds"), (-2, "element indices"),
                                       (-1, "at least 3 vertices")])
@pytest.mark.parametrize("column", [0, 2, 3])
def test_same_errors(bad, match, column):
    import torch

    import numba_celltree_amd as M

    v, f = polygons(4, 600, 5)
    tree = M.CellTree2d(v, f, -1)
    f = f.copy()
    f[431, column] = bad
    d_v, d_f = torch.from_numpy(v).cuda(), torch.from_numpy(f).cuda()
    if bad == -1 and column == 3:
        M.CellTree2d(d_v, d_f, -1)  # a fill value there is a triangle
        return
    with pytest.raises(ValueError, match=match):
        M.CellTree2d(d_v, d_f, -1)
    with pytest.raises(ValueError, match=match):
        tree.intersect_faces(d_v, d_f, -1)
    with pytest.raises(ValueError, match=match):
        M.CellTree2d(v, f, -1)
