"""The C entries with a flag per pair and the host list of a topology's left-over targets, which the package
itself no longer calls: the same as the mask forms and the device list it uses."""

import ctypes

import numpy as np
import pytest

from tests.test_gpu_subqueries import L, mesh, queries

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind", ["mixed", "hexagons"])
def test_flags_are_the_masks(kind):
    import torch

    import numba_celltree_amd as M
    from numba_celltree_amd import _device as D
    from numba_celltree_amd import _native

    tree = M.CellTree2d(*mesh(kind), -1)
    boxes = torch.from_numpy(queries(700, 5)[0]).cuda()
    ii, jj = tree._locate_boxes_dev(D.to_dev(boxes, torch.float64))
    n = int(ii.numel())
    area, keep = D.empty(n, torch.float64), D.empty(n, torch.int64)
    _native.call("ct_box_pairs", D.ptr(boxes), D.ptr(tree.d_vertices), D.ptr(tree.d_elements),
                 int(tree.d_elements.shape[1]), D.ptr(ii), D.ptr(jj), n, D.ptr(area), D.ptr(keep), D.stream())
    assert torch.equal(keep, (area > 0).long())
    offsets, total = D.exclusive_scan(keep)
    i, j, a = D.empty(total, torch.int64), D.empty(total, torch.int64), D.empty(total, torch.float64)
    _native.call("ct_compact_pairs", D.ptr(ii), D.ptr(jj), D.ptr(area), D.ptr(keep), D.ptr(offsets), n, D.ptr(i),
                 D.ptr(j), D.ptr(a), D.stream())
    for got, want in zip((i, j, a), tree.intersect_boxes(boxes)):
        assert torch.equal(got.view(torch.int64), want.view(torch.int64))


def test_rest_targets_of_the_host_list():
    import torch

    import numba_celltree_amd as M
    from numba_celltree_amd import _device as D
    from numba_celltree_amd import _native
    from numba_celltree_amd.regrid import RegridTopology

    tree = M.CellTree2d(*(torch.from_numpy(a).cuda() for a in mesh("mixed")), -1)
    tv, tf = mesh("hexagons")
    topo = RegridTopology(tree, torch.from_numpy(tv + 0.1 * L).cuda(), torch.from_numpy(tf).cuda(), -1)
    out, found = D.empty(topo.n_tgt, torch.int64), ctypes.c_int64(0)
    _native.call("ct_regrid_rest_targets", ctypes.byref(topo._struct), D.ptr(out), ctypes.byref(found), D.stream())
    assert 0 < found.value < topo.n_tgt
    assert np.array_equal(out[: found.value].cpu().numpy(), np.sort(topo.rest_targets.cpu().numpy()))
