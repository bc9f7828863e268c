"""CellTree2d on MI355X (drop-in for numba_celltree/celltree.py:37-351).

Construction and every query run as HIP kernels (libcelltree_hip.so): counter-clockwise
reordering, face bounding boxes, the level-synchronous tree build, traversals, the FP64
clippers and the barycentric weights.  Host inputs give host (numpy) outputs; device
tensors give device tensors.
"""

from typing import Optional, Tuple

import numpy as np
import torch

from numba_celltree_amd import _device as D
from numba_celltree_amd import _native
from numba_celltree_amd.cast import cast_bboxes, cast_edges, cast_faces, cast_vertices
from numba_celltree_amd.celltree_base import CellTree2dBase


class CellTree2d(CellTree2dBase):
    """
    Construct a cell tree from 2D vertices and a faces indexing array.

    Parameters
    ----------
    vertices: array of floats with shape ``(n_point, 2)`` (numpy or device tensor)
    faces: array of integers with shape ``(n_face, n_max_vert)``
    fill_value: int
        Fill value marking empty nodes in ``faces``.
    n_buckets: int, optional, default: 4 (2 .. 64)
    cells_per_leaf: int, optional, default: 2
    """

    def __init__(self, vertices, faces, fill_value: int, n_buckets: int = 4, cells_per_leaf: int = 2):
        if n_buckets < 2:
            raise ValueError("n_buckets must be >= 2")
        if cells_per_leaf < 1:
            raise ValueError("cells_per_leaf must be >= 1")
        vertices = cast_vertices(vertices, copy=True)
        d_vertices = D.to_dev(vertices, torch.float64) if D.is_device_tensor(faces) else None
        prep = None if d_vertices is None else D.prepare_faces(faces, fill_value, d_vertices, with_distances=True)
        if prep is not None:
            self._build_tree(d_vertices, prep.faces, prep.bb, n_buckets, cells_per_leaf, prep)
            return
        faces = cast_faces(faces, fill_value)
        d_vertices = D.to_dev(vertices, torch.float64)
        d_faces = D.faces_to_dev(faces, d_vertices.shape[0])
        n, nmax = int(d_faces.shape[0]), int(d_faces.shape[1])
        if n == 0:
            raise ValueError("faces is empty")
        if nmax < 3:
            raise ValueError("faces must have at least 3 columns")
        st = D.stream()
        _native.call("ct_counter_clockwise", D.ptr(d_vertices), D.ptr(d_faces), n, nmax, st)
        bb = D.empty((n, 4), torch.float64)
        _native.call("ct_build_face_bboxes", D.ptr(d_faces), n, nmax, D.ptr(d_vertices), D.ptr(bb), st)
        self._build_tree(d_vertices, d_faces, bb, n_buckets, cells_per_leaf)

    @property
    def faces(self) -> np.ndarray:
        """The counter-clockwise reordered faces (int64, fill -1)."""
        return self._elements_host()

    # ----------------------------------------------------------------- queries
    # Point batches at least this large, of a tree whose face rows and they multiply to at least
    # ORDERED_WORK, are processed in Morton order (ct_query_order, then ct_locate_points_in_order):
    # neighbouring lanes then share their root-to-leaf paths.  The sort takes 45 us and 7 ns per 1000
    # points; what it saves grows with the points and with what of the tree does not fit the L2s.  In
    # order / as they come, microseconds: 20,000 triangles, 2.6e5 points 79 / 33, 4e6 333 / 266;
    # 200,000 cells, 1e6 146 / 125, 4e6 359 / 414; a million cells, 2.6e5 96 / 61, 1e6 155 / 173,
    # 4e6 384 / 627.  ORDERED_MIN None: no batch is ordered; any other value than the default: it
    # alone decides.
    ORDERED_MIN = 3 << 18
    ORDERED_WORK = 1 << 40
    # Leaves of many cells: neighbours also share those, and points in no order leave the lanes of a
    # wavefront at different lengths of them, so from ORDERED_LEAF cells on the points and the cells of
    # a leaf decide, whatever the tree's size.  20,000 triangles, 8 cells a leaf, 2e6 216 / 213, 4e6
    # 355 / 377; 16 a leaf, 1e6 187 / 192, 1e7 886 / 1313; 64 a leaf, 2.7e5 218 / 226, 5e5 276 / 305
    # (a million cells 349 / 320 and 388 / 415); 130 a leaf, 2.7e5 329 / 366, 3e6 886 / 1750.
    ORDERED_LEAF = 8
    ORDERED_LEAF_MIN = 3 << 17       # half as many points where the product is twice as large
    ORDERED_LEAF_WORK = 1 << 24
    # Points whose gradients go to the vertices are put in order from this size on: it also lets the
    # backward add a face's points before it adds them to memory (1e6 points: 79 instead of 258 us).
    ORDERED_GRAD_MIN = 1 << 18

    def locate_points(self, points, tolerance: Optional[float] = None):
        """Index of the face containing each point, -1 outside (celltree.py:99-128)."""
        if tolerance is None:
            tolerance = self._default_tolerance()
        io = D.Io(points)
        pts = D.to_dev(cast_vertices(points), torch.float64)
        out = self._locate_points_dev(pts, float(tolerance))
        return io.out(out)

    def orders_points(self, n: int, vertex_gradients: bool = False) -> bool:
        """Whether a batch of n points is located in Morton order (``vertex_gradients``: as points
        whose weights take gradients to the vertices)."""
        if self.ORDERED_MIN is None or self.ORDERED_MIN != _ORDERED_MIN:
            return self.ORDERED_MIN is not None and n >= self.ORDERED_MIN
        leaf = int(self.cells_per_leaf)
        in_leaves = n * leaf // self.ORDERED_LEAF_WORK  # 0: too little, 2 and more: also for fewer points
        return (n >= self.ORDERED_MIN and n * int(self.d_elements.numel()) >= self.ORDERED_WORK
                or leaf >= self.ORDERED_LEAF and in_leaves > 0 and n >= self.ORDERED_LEAF_MIN // min(in_leaves, 2)
                or vertex_gradients and n >= self.ORDERED_GRAD_MIN)

    def _point_order(self, pts: torch.Tensor):
        """The Morton order of a point batch.  The order alone: writing the points in sorted order
        costs more in the sort (0.3 -> 0.8 ms at 1e7 points) than the contiguous read saves in the
        traversal."""
        return D.query_order(0, pts, self._bbox)

    def _locate_points_dev(self, pts: torch.Tensor, tolerance: float, order=None, sorted_pts=None) -> torch.Tensor:
        """``order`` / ``sorted_pts``: a processing order from ``D.query_order`` and, optionally,
        the points in that order (then read contiguously)."""
        n = int(pts.shape[0])
        out = D.empty(n, torch.int64)
        if order is None and self.orders_points(n):
            order = self._point_order(pts)
        if order is not None:
            _native.call("ct_locate_points_in_order", self.tree_ref, D.ptr(pts), n, D.ptr(order), D.ptr(sorted_pts),
                         tolerance, D.ptr(out), D.stream())
        else:
            _native.call("ct_locate_points", self.tree_ref, D.ptr(pts), n, tolerance, D.ptr(out), D.stream())
        return out

    def _locate_boxes_dev(self, d_boxes: torch.Tensor, prep=None):
        """``prep``: the faces (D.PreparedFaces) whose boxes these are; their index checks are made
        here, with the first value read back."""
        n = int(d_boxes.shape[0])
        st = D.stream()
        if self._gathers(n):
            return self._gather(1, d_boxes, self._gather_order(3, d_boxes), prep)
        order, srt = self._order(1, d_boxes)
        if prep is not None:
            prep.check(prep.checks[:3].tolist())
        if self._splits(n):
            return self._split_rows(1, d_boxes, order)[:2]
        counts = D.empty(n, torch.int64)
        hits, slots = self._hit_record(n, self.BOX_HIT_SLOTS, self.BOX_HIT_BUDGET)
        _native.call("ct_locate_boxes_count_rec", self.tree_ref, D.ptr(d_boxes), n, D.ptr(order), D.ptr(srt),
                     D.ptr(counts), D.ptr(hits), slots, st)
        offsets, total = D.exclusive_scan(counts)
        ii = D.empty(total, torch.int64)
        jj = D.empty(total, torch.int64)
        _native.call(
            "ct_locate_boxes_write_rec", self.tree_ref, D.ptr(d_boxes), n, D.ptr(order), D.ptr(srt),
            D.ptr(offsets), D.ptr(hits), slots, D.ptr(ii), D.ptr(jj), st,
        )
        return ii, jj

    def locate_boxes(self, bbox_coords) -> Tuple:
        """All (box, face) pairs whose bounding boxes strictly overlap (celltree.py:130-148)."""
        io = D.Io(bbox_coords)
        d_boxes = D.to_dev(cast_bboxes(bbox_coords), torch.float64)
        ii, jj = self._locate_boxes_dev(d_boxes)
        return io.out(ii), io.out(jj)

    @staticmethod
    def _kept(n: int):
        """(masks, counts) of a pair stage."""
        return D.empty((n + 63) // 64, torch.int64), D.empty((n + 63) // 64, torch.int64)

    def _compact(self, ii, jj, area, kept):
        masks, counts = kept
        offsets, total = D.exclusive_scan(counts)
        io_ = D.empty(total, torch.int64)
        jo = D.empty(total, torch.int64)
        ao = D.empty(total, torch.float64) if area is not None else None
        _native.call(
            "ct_compact_masks", D.ptr(ii), D.ptr(jj), D.ptr(area), D.ptr(masks), D.ptr(offsets),
            int(ii.numel()), D.ptr(io_), D.ptr(jo), D.ptr(ao), D.stream(),
        )
        return io_, jo, ao

    def intersect_boxes(self, bbox_coords) -> Tuple:
        """Box-face pairs with overlap area > 0 (celltree.py:150-184)."""
        io = D.Io(bbox_coords)
        d_boxes = D.to_dev(cast_bboxes(bbox_coords), torch.float64)
        ii, jj = self._locate_boxes_dev(d_boxes)
        n = int(ii.numel())
        area = D.empty(n, torch.float64)
        kept = self._kept(n)
        _native.call(
            "ct_box_pairs_masks", D.ptr(d_boxes), D.ptr(self.d_vertices), D.ptr(self.d_elements),
            int(self.d_elements.shape[1]), D.ptr(ii), D.ptr(jj), n, D.ptr(area), *(D.ptr(t) for t in kept), D.stream(),
        )
        i, j, a = self._compact(ii, jj, area, kept)
        return io.out(i), io.out(j), io.out(a)

    def _prepare_faces(self, d_vertices: torch.Tensor, d_faces: torch.Tensor) -> torch.Tensor:
        n, nmax = int(d_faces.shape[0]), int(d_faces.shape[1])
        st = D.stream()
        _native.call("ct_counter_clockwise", D.ptr(d_vertices), D.ptr(d_faces), n, nmax, st)
        bb = D.empty((n, 4), torch.float64)
        _native.call("ct_build_face_bboxes", D.ptr(d_faces), n, nmax, D.ptr(d_vertices), D.ptr(bb), st)
        return bb

    def _faces_in(self, vertices, faces, fill_value: int):
        """(vertices, faces, prepared faces or None) of a face query on the device; ``None``: the
        faces are checked but neither reordered nor boxed yet."""
        d_vertices = D.to_dev(cast_vertices(vertices), torch.float64)
        if D.is_device_tensor(faces) and faces.ndim == 2:
            # the check words lie behind the box query's offsets (_gather), read back together
            n = int(faces.shape[0])
            row = D.gather_row(n)
            prep = D.prepare_faces(faces, fill_value, d_vertices, with_distances=False, checks=row[n + 1: n + 9])
            if prep is not None:
                prep.row = row
                return d_vertices, prep.faces, prep
        return d_vertices, D.faces_to_dev(cast_faces(faces, fill_value), d_vertices.shape[0]), None

    def _face_pairs(self, d_vertices, d_faces, with_area: bool, prep=None):
        """locate_boxes on the faces' bboxes, then the fused SAT (+ clip area) pair stage."""
        bb = self._prepare_faces(d_vertices, d_faces) if prep is None else prep.bb
        ii, jj = self._locate_boxes_dev(bb, prep)
        n = int(ii.numel())
        area = D.empty(n, torch.float64) if with_area else None
        kept = self._kept(n)
        _native.call(
            "ct_face_pairs_masks", D.ptr(d_vertices), D.ptr(d_faces), int(d_faces.shape[1]),
            D.ptr(self.d_vertices), D.ptr(self.d_elements), int(self.d_elements.shape[1]),
            D.ptr(ii), D.ptr(jj), n, int(with_area), D.ptr(area), *(D.ptr(t) for t in kept), D.stream(),
        )
        return self._compact(ii, jj, area, kept)

    def locate_faces(self, vertices, faces) -> Tuple:
        """Face pairs that intersect or touch (SAT), celltree.py:186-226.

        As in the reference, a host ``faces`` array is reordered counter-clockwise in place.
        """
        io = D.Io(vertices, faces)
        d_vertices = D.to_dev(cast_vertices(vertices), torch.float64)
        d_faces = D.faces_to_dev(faces, d_vertices.shape[0])
        i, j, _ = self._face_pairs(d_vertices, d_faces, with_area=False)
        if isinstance(faces, np.ndarray) and faces.ndim == 2:
            faces[...] = d_faces.cpu().numpy().astype(faces.dtype)
        elif isinstance(faces, torch.Tensor) and faces.is_cuda and faces.dtype == torch.int32:
            faces.copy_(d_faces)
        return io.out(i), io.out(j)

    def intersect_faces(self, vertices, faces, fill_value: int) -> Tuple:
        """Face pairs with overlap area > 0, and the area (celltree.py:228-269)."""
        io = D.Io(vertices, faces)
        d_vertices, d_faces, prep = self._faces_in(vertices, faces, fill_value)
        i, j, a = self._face_pairs(d_vertices, d_faces, True, prep)
        return io.out(i), io.out(j), io.out(a)

    def intersect_edges(self, edge_coords) -> Tuple:
        """Clipped sub-segment of every segment inside every face, ordered along each
        segment (celltree.py:271-304)."""
        io = D.Io(edge_coords)
        d_edges = D.to_dev(cast_edges(edge_coords), torch.float64)
        ii, jj, xy = self._locate_edges(d_edges, 1)
        return io.out(ii), io.out(jj), io.out(xy)

    def compute_barycentric_weights(self, points, tolerance: Optional[float] = None) -> Tuple:
        """Face index and barycentric weights of each point (celltree.py:306-351):
        Wachspress weights when faces have more than 3 columns, else triangle weights."""
        if tolerance is None:
            tolerance = self._default_tolerance()
        io = D.Io(points)
        pts = D.to_dev(cast_vertices(points), torch.float64)
        n = int(pts.shape[0])
        nmax = int(self.d_elements.shape[1])
        face = D.empty(n, torch.int64)
        w = D.empty((n, nmax), torch.float64)
        _native.call(
            "ct_compute_barycentric_weights", self.tree_ref, D.ptr(pts), n, float(tolerance),
            D.ptr(face), D.ptr(w), D.stream(),
        )
        return io.out(face), io.out(w)


_ORDERED_MIN = CellTree2d.ORDERED_MIN
