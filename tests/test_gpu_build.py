"""The tree build against the oracle where its stages meet: the cell counts at which a node goes
from the level-by-level kernels to one workgroup (1024, 512, 256 and 128 cells by bucket count),
tiles of 1024 cells, leaves larger than a workgroup's subtree, nodes that retry or stay degenerate
leaves, and trees too unbalanced for the levels launched ahead.  Nodes and order are compared bit
for bit; the node boxes of the build with those of ct_node_boxes."""

import ctypes

import numpy as np
import pytest

from numba_celltree_amd import synthetic as S
from oracle import refcpu as R

pytestmark = pytest.mark.gpu


def check(v, f, n_buckets=4, cells_per_leaf=2):
    import torch

    import numba_celltree_amd as M
    from numba_celltree_amd import _device as D
    from numba_celltree_amd import _native

    g = M.CellTree2d(v, f, -1, n_buckets=n_buckets, cells_per_leaf=cells_per_leaf)
    o = R.OracleCellTree2d(v, f, -1, n_buckets=n_buckets, cells_per_leaf=cells_per_leaf)
    gn, on = g.nodes, o.nodes
    assert gn.shape == on.shape
    for field in ("child", "ptr", "size", "dim"):
        assert np.array_equal(gn[field], on[field]), field
    for field in ("Lmax", "Rmin"):
        assert np.array_equal(gn[field].view(np.int64), on[field].view(np.int64)), field
    assert np.array_equal(g.bb_indices, o.bb_indices)
    assert np.array_equal(g.bbox, o.bbox)
    assert np.array_equal(g.bb_distances, o.bb_distances)
    depth = np.zeros(len(on), dtype=int)
    for x in range(len(on)):
        c = on["child"][x]
        if c >= 0:
            depth[c] = depth[c + 1] = depth[x] + 1
    assert g.depth == depth.max()
    boxes = torch.empty_like(g.d_node_boxes)
    scratch = torch.empty(g.n_nodes, dtype=torch.int32, device="cuda")
    _native.call("ct_node_boxes", g.tree_ref, D.ptr(scratch), D.ptr(boxes), D.stream())
    a, b = g.d_node_boxes[1:], boxes[1:]
    assert torch.equal(torch.isnan(a), torch.isnan(b))
    assert torch.equal(torch.nan_to_num(a), torch.nan_to_num(b))
    # the one-call form, into arrays of the pessimistic capacity
    L = _native.lib()
    n = len(f)
    ws = D.empty(int(L.ct_build_workspace_bytes(n, n_buckets)), torch.uint8)
    nodes = D.empty(32 * int(L.ct_max_nodes(n)), torch.uint8)
    order = D.empty(n, torch.int32)
    n_nodes, d = ctypes.c_int64(0), ctypes.c_int32(0)
    _native.call("ct_build", D.ptr(g.d_bb_coords), n, n_buckets, cells_per_leaf, D.ptr(ws), ws.numel(), D.ptr(nodes),
                 D.ptr(order), ctypes.byref(n_nodes), ctypes.byref(d), D.stream())
    assert (n_nodes.value, d.value) == (g.n_nodes, g.depth)
    assert torch.equal(nodes[: 32 * g.n_nodes], g.d_nodes) and torch.equal(order, g.d_bb_indices)


@pytest.fixture(scope="module")
def mesh():
    return S.jittered_grid(61, 10.0, 0.3, 1.0, 11)  # 7200 triangles


@pytest.mark.parametrize("n", [1, 2, 3, 5, 64, 1023, 1024, 1025, 1026, 2047, 2049, 3073, 7200])
@pytest.mark.parametrize("cells_per_leaf", [1, 2])
def test_sizes_around_the_stages(mesh, n, cells_per_leaf):
    v, f = mesh
    check(v, f[np.random.default_rng(n).permutation(len(f))[:n]], 4, cells_per_leaf)


@pytest.mark.parametrize("n_buckets,n", [(2, 1025), (3, 4000), (5, 2050), (8, 7200), (9, 513), (16, 7200), (17, 257),
                                         (32, 3000), (33, 129), (63, 1500), (64, 7200)])
@pytest.mark.parametrize("cells_per_leaf", [1, 3])
def test_bucket_classes(mesh, n_buckets, n, cells_per_leaf):
    v, f = mesh
    check(v, f[:n], n_buckets, cells_per_leaf)


@pytest.mark.parametrize("cells_per_leaf", [700, 1024, 1025, 3000, 8000])
def test_leaves_larger_than_a_subtree(mesh, cells_per_leaf):
    check(*mesh, 4, cells_per_leaf)


@pytest.mark.parametrize("copies,n_buckets", [(3, 4), (1500, 4), (5000, 64)])
def test_identical_cells_stay_one_leaf(mesh, copies, n_buckets):
    """Cells that share a centroid land in one bucket in both dimensions: a leaf of any size,
    beside ordinary ones."""
    v, f = mesh
    check(v, np.concatenate([f[:900], np.repeat(f[2000:2001], copies, axis=0)]), n_buckets, 2)


def test_one_row_of_cells_retries():
    """Cells in one row: every split along y retries along x."""
    x = np.arange(3001.0)
    v = np.concatenate([np.column_stack([x, 0 * x]), np.column_stack([x, 0 * x + 1.0])])
    i = np.arange(3000)
    check(v, np.column_stack([i, i + 1, i + 3002, i + 3001]).astype(np.int32))


@pytest.mark.parametrize("levels", [250, 600])
def test_unbalanced_trees_need_more_levels(levels):
    """A few cells leave the large node per level: many more levels than a balanced tree's."""
    check(*S.graded_corner(levels))


@pytest.mark.parametrize("n", [900, 5000])
def test_nan_cells_raise_index_error(mesh, n):
    import numba_celltree_amd as M

    v, f = mesh
    v = v.copy()
    v[f[n // 2]] = np.nan
    with pytest.raises(IndexError, match="degenerate bucketing"):
        M.CellTree2d(v, f[:n], -1)
