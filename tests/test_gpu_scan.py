"""ct_exclusive_scan at the sizes where it changes its launches (one workgroup up to 8192 elements, carries
added up by every workgroup up to 1024 tiles of 2048), against torch.cumsum: whole numbers, equal."""

import pytest

pytestmark = pytest.mark.gpu

FOLD = 1024 * 2048


@pytest.mark.parametrize("n", [0, 1, 7, 8, 9, 8191, 8192, 8193, 10_241, FOLD - 1, FOLD, FOLD + 1, 3 * FOLD + 5])
def test_exclusive_scan(n):
    import torch

    from numba_celltree_amd import _device as D

    g = torch.Generator(device="cuda").manual_seed(n)
    counts = torch.randint(0, 1 << 33, (n,), generator=g, device="cuda", dtype=torch.int64)
    offsets, total = D.exclusive_scan(counts)
    want = torch.zeros(n + 1, dtype=torch.int64, device="cuda")
    torch.cumsum(counts, 0, out=want[1:])
    assert torch.equal(offsets[: n + 1], want) and total == int(want[-1])
