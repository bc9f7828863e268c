"""The lists of a regridding (ct_regrid_lists): the pairs of every source, the corners of every vertex,
the first pair of every target and the targets a block of pairs does not hold, against numpy: lists
from empty to longer than a wavefront and a workgroup sort (a vertex of a fan has as many corners as
the mesh has faces, one large source cell meets every target)."""

import numpy as np
import pytest

from numba_celltree_amd import synthetic as S

pytestmark = pytest.mark.gpu


def fan(n: int):
    """n thin triangles around the origin, n shared vertices on the circle."""
    a = np.linspace(0.0, 2.0 * np.pi, n, endpoint=False)
    v = np.concatenate([[[0.0, 0.0]], np.stack([np.cos(a), np.sin(a)], axis=1)])
    k = np.arange(n)
    return v, np.stack([np.zeros(n, np.int64), k + 1, (k + 1) % n + 1], axis=1)


def square(lo: float, hi: float):
    return np.array([[lo, lo], [hi, lo], [hi, hi], [lo, hi]]), np.array([[0, 1, 2, 3]])


def grouped(key, n_keys):
    order = np.argsort(key, kind="stable")
    return np.searchsorted(key[order], np.arange(n_keys + 1)), order


def cases():
    grid = S.jittered_grid(30, 2.0, 0.2, 0.5, 1)
    grid = (grid[0] - 1.0, grid[1])
    hexagons = S.hex_voronoi(20, 20, 2.0, 0.1, 2)
    hexagons = (hexagons[0] - 1.0, hexagons[1])
    yield "grids", grid, hexagons
    yield "away", grid, square(5.0, 6.0)
    for n in (3, 63, 64, 65, 129, 1000, 1025, 8192, 8193, 20_000):
        yield f"fan{n}", fan(n), square(-0.4, 0.5)
        if n in (65, 1025, 8193, 20_000):
            yield f"onto_fan{n}", square(-2.0, 2.0), fan(n)


@pytest.mark.parametrize("name, src, tgt", list(cases()), ids=lambda x: x if isinstance(x, str) else "")
def test_lists(name, src, tgt):
    import torch

    import numba_celltree_amd as M
    from numba_celltree_amd.regrid import Regridder

    tree = M.CellTree2d(torch.from_numpy(src[0]).cuda(), torch.from_numpy(src[1]).cuda(), -1)
    t = Regridder(tree, torch.from_numpy(tgt[0]).cuda(), torch.from_numpy(tgt[1]).cuda()).topology
    tt, ss = t.tt.cpu().numpy(), t.ss.cpu().numpy()
    assert (np.diff(tt) >= 0).all()
    off = np.searchsorted(tt, np.arange(t.n_tgt + 1))
    assert np.array_equal(t.tgt_offsets.cpu().numpy(), off)
    soff, perm = grouped(ss, t.n_src)
    assert np.array_equal(t.src_offsets.cpu().numpy(), soff)
    assert np.array_equal(t.perm_by_src.cpu().numpy(), perm)
    assert np.array_equal(t.src_tgt.cpu().numpy(), tt[perm])
    for mesh, n_v in (("tgt", t.n_tgt_vertices), ("src", t.n_src_vertices)):
        flat = getattr(t, f"{mesh}_faces").cpu().numpy().reshape(-1)
        ids = np.flatnonzero(flat >= 0)
        voff, order = grouped(flat[ids], n_v)
        assert np.array_equal(getattr(t, f"{mesh}_vertex_offsets").cpu().numpy(), voff)
        assert np.array_equal(getattr(t, f"{mesh}_vertex_corners").cpu().numpy(), ids[order])
    b, e = off[:-1], off[1:]
    rest = np.flatnonzero((e == b) | (b // 256 != (e - 1) // 256))
    assert np.array_equal(np.sort(t.rest_targets.cpu().numpy()), rest)
