"""Sizes ct_regrid_lists takes, by the checks it makes before any device work: a group of items below 2^31, and
together more than 2^32 - 1 (pairs and corners that a 32-bit launch does not hold at once)."""

import ctypes

import pytest


def status(n_pairs, n_tgt, n_src, n_max=4):
    from numba_celltree_amd import _native

    t = _native.CtRegridTopology()
    for name in ("tgt_faces", "src_faces", "tt", "ss"):
        setattr(t, name, 32)  # never read: no workspace is given
    t.n_pairs, t.n_tgt, t.n_src, t.n_tgt_vertices, t.n_src_vertices = n_pairs, n_tgt, n_src, max(n_tgt, 1), n_src
    t.n_max_t = t.n_max_s = n_max
    return _native.lib().ct_regrid_lists(ctypes.byref(t), None, 0, *([32] * 10), None)


@pytest.mark.parametrize("n_pairs, n_tgt, n_src, taken", [
    (1000, 10, 10, True),
    ((1 << 31) - 1, 1 << 28, 1 << 28, True),           # 2^32 - 1 items
    ((1 << 31) - 1, (1 << 29) - 1, (1 << 29) - 1, True),  # some 3 * 2^31
    (1 << 31, 10, 10, False),
    (1000, 1 << 29, 10, False),
    (1000, 10, 1 << 29, False),
])
def test_sizes(n_pairs, n_tgt, n_src, taken):
    from numba_celltree_amd import _native

    assert status(n_pairs, n_tgt, n_src) == (_native.CT_ERR_WORKSPACE if taken else _native.CT_ERR_ARG)
