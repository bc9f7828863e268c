"""Device plumbing: torch tensors hold every device array, the HIP library computes.

Inputs may be host arrays (numpy / lists) or device tensors.  ``Io`` remembers which kind
came in so results go back the same way: numpy in, numpy out (the reference's contract);
device tensor in, device tensor out (no PCIe round trip).
"""

import ctypes
import warnings

import numpy as np
import torch

from numba_celltree_amd import _native
from numba_celltree_amd.constants import NodeDType


def device() -> torch.device:
    # Every array of a call asks for this: is_available() counts the devices anew each time.
    if not torch.cuda.is_initialized() and not torch.cuda.is_available():
        raise RuntimeError(
            "numba_celltree_amd computes on a ROCm GPU only, and none is visible "
            "(torch.cuda.is_available() is False)"
        )
    return torch.device("cuda", torch.cuda.current_device())


def stream() -> int:
    """The current stream's handle (without torch.cuda.current_stream()'s Stream object)."""
    return torch._C._cuda_getCurrentRawStream(torch.cuda.current_device())


def ptr(t) -> int:
    return 0 if t is None else t.data_ptr()


def is_device_tensor(x) -> bool:
    return isinstance(x, torch.Tensor) and x.is_cuda


class Io:
    """Tracks whether a call received device tensors, and converts results back."""

    def __init__(self, *inputs):
        self.device_io = any(is_device_tensor(x) for x in inputs)

    def out(self, t: torch.Tensor):
        if self.device_io:
            return t
        return t.cpu().numpy()


def host_tensor(a: np.ndarray) -> torch.Tensor:
    """A CPU tensor sharing ``a``'s memory; read-only arrays (views of immutable bytes) are
    shared too, for copies that only read them."""
    a = np.ascontiguousarray(a)
    if a.flags.writeable:
        return torch.from_numpy(a)
    with warnings.catch_warnings():
        warnings.filterwarnings("ignore", message="The given NumPy array is not writable")
        return torch.from_numpy(a)


def to_dev(x, dtype: torch.dtype) -> torch.Tensor:
    """Contiguous, 32-byte aligned device tensor of ``dtype`` (copies host data).

    The kernels read points, boxes and segments with 16- and 32-byte vector loads; a view
    that starts mid-row is copied to a fresh (aligned) allocation.
    """
    dev = device()
    if isinstance(x, torch.Tensor):
        t = (x if x.dtype == dtype and x.device == dev else x.to(device=dev, dtype=dtype)).contiguous()
    else:
        t = host_tensor(np.asarray(x)).to(device=dev, dtype=dtype).contiguous()
    if t.data_ptr() % 32:
        t = t.clone()
    return t


def faces_to_dev(faces, n_vertices: int, allow_fill: bool = True) -> torch.Tensor:
    """int32 device copy of a (n, n_max_vert) index array.

    Every index must address one of ``n_vertices`` vertices; -1 (the fill value) is allowed
    only where ``allow_fill`` (face rows, past their first 3 entries; edge rows have no
    fill).  The kernels read vertices without bounds checks, so this is checked here, before
    any launch."""
    if isinstance(faces, torch.Tensor):
        f = faces
    else:
        f = host_tensor(np.asarray(faces))
    if f.numel():
        # one host round trip for all three checks (a device tensor costs a synchronization
        # per value read back)
        lo, hi = torch.aminmax(f)
        first3 = allow_fill and f.ndim == 2 and f.shape[1] >= 3
        lo3 = f[:, :3].amin() if first3 else lo
        hi, lo, lo3 = (int(v) for v in torch.stack([hi, lo, lo3]).tolist())
        check_indices(hi, lo, lo3 if first3 else 0, n_vertices, allow_fill)
    return f.to(device=device(), dtype=torch.int32).contiguous()


def check_indices(hi: int, lo: int, lo3: int, n_vertices: int, allow_fill: bool = True) -> None:
    """Raises unless the largest (hi), smallest (lo) and smallest first-three-columns (lo3) index
    of an element array address ``n_vertices`` vertices."""
    if hi >= min(int(n_vertices), 2**31):
        raise ValueError(f"element index {hi} is out of bounds for {int(n_vertices)} vertices")
    if lo < (-1 if allow_fill else 0):
        what = "[-1, n_vertices)" if allow_fill else "[0, n_vertices)"
        raise ValueError(f"element indices must lie in {what}, found {lo}")
    if lo3 < 0:
        # polygon_length (geometry_utils.py:72-79) takes the first 3 entries as vertices
        raise ValueError("every face needs at least 3 vertices (a fill value among its first 3 entries)")


class PreparedFaces:
    """Device face rows made ready by ct_prepare_faces: ``faces`` (int32, counter-clockwise), ``bb``
    (their boxes), ``distances`` (when asked for) and ``checks`` (8 device words; ``check`` raises what
    ``faces_to_dev`` raises once they are on the host)."""

    def __init__(self, faces, bb, distances, checks, n_vertices):
        self.faces, self.bb, self.distances, self.checks, self.n_vertices = faces, bb, distances, checks, n_vertices

    def check(self, words) -> None:
        """``words``: the first three of ``checks`` as host integers (int64 bit patterns)."""
        raw = (ctypes.c_uint64 * 3)(*[int(w) & 0xFFFFFFFFFFFFFFFF for w in words[:3]])
        out = (ctypes.c_int64 * 3)()
        _native.call("ct_check_values", raw, out)
        check_indices(out[0], out[1], out[2], self.n_vertices)


def prepare_faces(faces, fill_value, d_vertices: torch.Tensor, with_distances: bool, checks=None):
    """The rows of a device index array in one pass (PreparedFaces; the index checks are the
    caller's, after its next synchronization), or None where that pass does not apply: host
    arrays, another device, no faces or vertices, fewer than 3 or more than 8 columns, a fill value
    that is no integer.  ``checks``: 8 int64 to use for the check words."""
    if not is_device_tensor(faces) or faces.device != device() or faces.ndim != 2:
        return None
    n, nmax = int(faces.shape[0]), int(faces.shape[1])
    nv = int(d_vertices.shape[0])
    if n == 0 or nv == 0 or not 3 <= nmax <= 8 or faces.is_complex():
        return None
    try:
        fill = int(fill_value)
    except (TypeError, ValueError, OverflowError):
        return None
    if fill != fill_value or not -(2**63) <= fill < 2**63:
        return None
    if faces.dtype not in (torch.int32, torch.int64):
        faces = faces.to(torch.int64)
    faces = faces.contiguous()
    out = empty((n, nmax), torch.int32)
    bb = empty((n, 4), torch.float64)
    distances = empty((n, 3), torch.float64) if with_distances else None
    if checks is None:
        checks = empty(8, torch.int64)
    _native.call("ct_prepare_faces", ptr(faces), faces.element_size(), n, nmax, fill, nv, ptr(d_vertices), ptr(out),
                 ptr(bb), ptr(distances), ptr(checks), stream())
    return PreparedFaces(out, bb, distances, checks, nv)


def index_to_dev(x, n: int, allow_missing: bool = False) -> torch.Tensor:
    """int64 device copy of an index array into n items (-1 allowed where ``allow_missing``)."""
    t = x if isinstance(x, torch.Tensor) else torch.from_numpy(np.ascontiguousarray(x))
    if t.numel():
        lo, hi = (int(v) for v in torch.stack(torch.aminmax(t)).tolist())  # one host round trip
        if hi >= int(n) or lo < (-1 if allow_missing else 0):
            raise ValueError(f"indices must lie in [{-1 if allow_missing else 0}, {int(n)}), found [{lo}, {hi}]")
    return to_dev(t, torch.int64)


def empty(shape, dtype) -> torch.Tensor:
    return torch.empty(shape, dtype=dtype, device=device())


def gather_row(n: int) -> torch.Tensor:
    """The int64 words of a ct_gather_* call on n queries: n + 1 offsets, 8 check words
    (PreparedFaces), the working words."""
    return empty(n + 9 + int(_native.lib().ct_gather_tail_words()), torch.int64)


def exclusive_scan(counts: torch.Tensor, total: bool = True, offsets=None):
    """Offsets (n + 1, int64, device) of ``counts`` and the total (host int: synchronizes;
    None with ``total=False``).  ``offsets``: n + 1 or more int64 to write them to."""
    n = counts.numel()
    if offsets is None:
        offsets = empty(n + 1, torch.int64)
    ws = empty(int(_native.lib().ct_scan_workspace_bytes(n)), torch.uint8)
    _native.call("ct_exclusive_scan", ptr(counts), n, ptr(offsets), ptr(ws), ws.numel(), stream())
    return offsets, (int(offsets[n].item()) if total else None)


def query_order(kind: int, queries: torch.Tensor, bbox, with_sorted: bool = False):
    """Processing order (int32, device) of n queries: kind 0 points, 1 boxes, 2 segments.
    With ``with_sorted``, returns (order, sorted) where sorted[i] = queries[order[i]]."""
    n = int(queries.shape[0])
    order = empty(n, torch.int32)
    sorted_q = empty((n, 2 if kind == 0 else 4), torch.float64) if with_sorted else None
    ws = empty(int(_native.lib().ct_order_workspace_bytes(n)), torch.uint8)
    bb = (ctypes.c_double * 4)(*[float(x) for x in bbox])
    _native.call("ct_query_order", kind, ptr(queries), n, bb, ptr(ws), ws.numel(), ptr(order), ptr(sorted_q),
                 stream())
    return (order, sorted_q) if with_sorted else order


# ------------------------------------------------------------------ node records
def nodes_to_host(raw: torch.Tensor, n_nodes: int) -> np.ndarray:
    """Device ``ct_node`` bytes -> the reference's packed NodeDType array."""
    buf = raw[: 32 * n_nodes].cpu().numpy()
    f = buf.view(np.float64).reshape(n_nodes, 4)
    i = buf.view(np.int32).reshape(n_nodes, 8)
    out = np.empty(n_nodes, dtype=NodeDType)
    out["child"] = i[:, 4]
    out["Lmax"] = f[:, 0]
    out["Rmin"] = f[:, 1]
    out["ptr"] = i[:, 5]
    out["size"] = i[:, 6]
    out["dim"] = i[:, 7] != 0
    return out


def nodes_to_device(nodes: np.ndarray) -> torch.Tensor:
    """NodeDType array -> device ``ct_node`` bytes."""
    n = len(nodes)
    buf = np.zeros(32 * n, dtype=np.uint8)
    f = buf.view(np.float64).reshape(n, 4)
    i = buf.view(np.int32).reshape(n, 8)
    f[:, 0] = nodes["Lmax"]
    f[:, 1] = nodes["Rmin"]
    i[:, 4] = nodes["child"]
    i[:, 5] = nodes["ptr"]
    i[:, 6] = nodes["size"]
    i[:, 7] = nodes["dim"].astype(np.int32)
    return torch.from_numpy(buf).to(device())
