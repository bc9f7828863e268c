"""The work that users of this package have it do, as measured cases.

A user holds meshes and queries on the GPU and calls the tree's constructor, its query methods, the
regridder, the differentiable weights and the many-mesh batch.  Every mesh here is synthetic, of the
kinds the repository's benchmark and tests use: a jittered vertex grid split into triangles, a mix
of triangles and quadrilaterals in random order, and a honeycomb of hexagons.  Everything is drawn
on the GPU from the seed.  How many rows a query returns and how many nodes a tree has follows from
the geometry, and the outputs of one case have one shape: there the geometry is the case's own, and
the seed gives its pose (a quarter turn and a power-of-two scale, both exact) and the order of faces
and queries; elsewhere the seed gives the geometry too.

A case is a dict: ``op`` names the call, ``kind`` and ``cells`` the tree's mesh, the rest the
queries.  ``exact`` restates the real-valued results with plain torch in 64 bits: bounding boxes,
clipped segments, barycentric weights with their gradients, and the regridded fields with theirs.
Cell indices are whole numbers and have no such value; overlap areas come in the order in which the
tree's walk meets the pairs, which nothing outside the package can lay out.
"""

import math

import torch

from numba_celltree_amd import CellTree2d
from numba_celltree_amd.barycentric import barycentric_weights
from numba_celltree_amd.batch import BatchGraph, TreeBatch, concat_queries
from numba_celltree_amd.regrid import Regridder

LENGTH = 1000.0   # side of the square every mesh covers
BOX_LO, BOX_HI = 0.1, 20.0    # box widths and heights, log-uniform, in cell sides
SEG_LO, SEG_HI = 0.1, 50.0    # segment lengths, log-uniform, in cell sides
JITTER = 0.25                 # vertices move by up to this share of the grid spacing


# ------------------------------------------------------------------------------------ cases
def listed():
    return [
        # One small model domain: the tree is built when it is loaded, and again for each one of many.
        {"name": "build_20k", "op": "build", "kind": "triangles", "cells": 20_000, "n_buckets": 4, "cells_per_leaf": 2},
        # A national or continental mesh: the build a program pays at its start or after a mesh change.
        {"name": "build_1m", "op": "build", "kind": "mixed", "cells": 1_000_000, "n_buckets": 4, "cells_per_leaf": 2},
        # Some stations looked up in a small mesh: one launch, latency alone.
        {"name": "points_1k", "op": "points", "kind": "triangles", "cells": 20_000, "queries": 1_000},
        # The repository's headline: the pixels or particles of a large model, in no order.
        {"name": "points_10m", "op": "points", "kind": "mixed", "cells": 1_000_000, "queries": 10_000_000},
        # Raster cells or tiles of mixed sizes against a large mesh.
        {"name": "boxes_1m", "op": "boxes", "kind": "mixed", "cells": 1_000_000, "queries": 1_000_000},
        # A river or road network over one of many medium meshes: a ragged handful of segments.
        {"name": "segments_2k", "op": "segments", "kind": "mixed", "cells": 45_000, "queries": 1_999},
        # A dense line network over the large mesh.
        {"name": "segments_1m", "op": "segments", "kind": "mixed", "cells": 1_000_000, "queries": 1_000_000},
        # Overlap areas of two unstructured meshes, the conservative coupling of two models.
        {"name": "faces_250k", "op": "faces", "kind": "triangles", "cells": 1_000_000, "targets": 250_000},
        # A regridder made for a new pair of meshes, with its sparse operator (odd sizes).
        {"name": "regrid_setup_61k", "op": "regrid_setup", "kind": "mixed", "cells": 180_000, "targets": 61_009},
        # A training or assimilation step through the regridder: 16 fields, gradients of all three inputs.
        {"name": "regrid_grad_16f", "op": "regrid_grad", "kind": "mixed", "cells": 1_000_000, "targets": 250_000,
         "fields": 16},
        # Interpolation weights at many points and their gradients in the points and the mesh.
        {"name": "barycentric_grad_1m", "op": "barycentric_grad", "kind": "triangles", "cells": 20_000,
         "queries": 1_000_000},
        # Many domains of very different sizes in one graph: points and segments of each.
        {"name": "batch_32", "op": "batch", "kind": "mixed", "cells": 200_000, "meshes": 32},
    ]


def _between(rng, lo, hi):
    """A whole number between lo and hi, spread evenly over their logarithm."""
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    op = rng.choice(["build", "points", "boxes", "segments", "faces", "regrid_setup", "regrid_grad", "barycentric_grad",
                     "batch"])
    kind = rng.choice(["triangles", "mixed", "mixed", "hexagons"])
    cells = _between(rng, 1_000, 1_000_000)
    case = {"op": op, "kind": kind, "cells": cells}
    if op == "build":
        case.update(n_buckets=rng.choice([2, 4, 4, 4, 8]), cells_per_leaf=rng.choice([1, 2, 2, 2, 4]))
    elif op == "points":
        case.update(queries=_between(rng, 100, 10_000_000))
    elif op in ("boxes", "segments"):
        case.update(queries=_between(rng, 100, 1_000_000))
    elif op == "batch":
        case.update(kind="mixed", cells=_between(rng, 20_000, 200_000), meshes=rng.randint(4, 32))
    elif op == "barycentric_grad":
        case.update(kind="triangles", queries=_between(rng, 1_000, 1_000_000))
    else:
        if op == "regrid_setup":
            cells = case["cells"] = _between(rng, 1_000, 250_000)
        case.update(kind=rng.choice(["triangles", "mixed"]), targets=max(64, _between(rng, cells / 16, cells / 2.5)))
        if op == "regrid_grad":
            case["cells"] = min(case["cells"], 1_000_000)
            case.update(targets=min(case["targets"], 250_000), fields=rng.choice([1, 3, 8, 16]))
    return case


# ------------------------------------------------------------------------------------ meshes
def _generator(seed, salt):
    return torch.Generator(device="cuda").manual_seed((int(seed) * 1_000_003 + salt) % (1 << 62))


def _uniform(g, lo, hi, *shape):
    return torch.rand(*shape, generator=g, device="cuda", dtype=torch.float64) * (hi - lo) + lo


class _Pose:
    """A quarter turn about the origin and a power-of-two scale: exact in floating point, so that the
    posed geometry has the same overlaps.  A tree's splits follow the axes, so a build is not turned."""

    def __init__(self, seed, turn=True):
        g = torch.Generator().manual_seed(int(seed) % (1 << 62) + 17)
        self.scale = 2.0 ** int(torch.randint(-3, 4, (1,), generator=g))
        self.turns = int(torch.randint(0, 4, (1,), generator=g)) if turn else 0

    def xy(self, a):
        x, y = a[..., 0] * self.scale, a[..., 1] * self.scale
        for _ in range(self.turns):
            x, y = -y, x
        return torch.stack([x, y], dim=-1).contiguous()

    def boxes(self, b):
        lo, hi = self.xy(b[:, 0::2]), self.xy(b[:, 1::2])
        lo, hi = torch.minimum(lo, hi), torch.maximum(lo, hi)
        return torch.stack([lo[:, 0], hi[:, 0], lo[:, 1], hi[:, 1]], dim=1).contiguous()


def _in_order(faces, seed, shuffle):
    """The faces in an order of the seed's: any (a mesh from a generator that shuffles), or one that keeps
    neighbours together, begun at another face."""
    g = _generator(seed, 8)
    if shuffle:
        return faces[torch.randperm(faces.shape[0], generator=g, device="cuda")].contiguous()
    return torch.roll(faces, int(torch.randint(0, faces.shape[0], (1,), generator=g, device="cuda")), dims=0).contiguous()


def _grid_mesh(cells, split, seed):
    """(vertices, faces): a jittered vertex grid whose quads are split into two triangles with share
    ``split``; all faces counter-clockwise, -1 behind a triangle of a mixed mesh."""
    nq = max(2, int(round(math.sqrt(cells / (1.0 + split)))))
    nv, h = nq + 1, LENGTH / nq
    g = _generator(seed, 1)
    line = torch.arange(nv, device="cuda", dtype=torch.float64) * h
    line[-1] = LENGTH
    y, x = torch.meshgrid(line, line, indexing="ij")
    xy = torch.stack([x, y], dim=-1)
    move = _uniform(g, -JITTER * h, JITTER * h, nv, nv, 2)
    xy[1:-1, 1:-1] += move[1:-1, 1:-1]
    ids = torch.arange(nv * nv, device="cuda", dtype=torch.int32).reshape(nv, nv)
    quads = torch.stack([ids[:-1, :-1], ids[:-1, 1:], ids[1:, 1:], ids[1:, :-1]], dim=-1).reshape(-1, 4)
    if split >= 1.0:
        faces = torch.stack([quads[:, [0, 1, 2]], quads[:, [0, 2, 3]]], dim=1).reshape(-1, 3)
    else:
        cut = torch.randperm(nq * nq, generator=g, device="cuda") < int(round(split * nq * nq))
        tri = torch.full((int(cut.sum()), 2, 4), -1, dtype=torch.int32, device="cuda")
        tri[:, 0, :3] = quads[cut][:, [0, 1, 2]]
        tri[:, 1, :3] = quads[cut][:, [0, 2, 3]]
        faces = torch.cat([quads[~cut], tri.reshape(-1, 4)])
    return xy.reshape(-1, 2).contiguous(), faces.contiguous()


def _hexagons(cells, seed):
    """(vertices, faces): a honeycomb of about ``cells`` hexagons over the square, its border cells
    sticking out a little, vertices moved by a tenth of a side."""
    n = max(2, int(round(math.sqrt(cells))))
    dx, dy = LENGTH / n, LENGTH / n
    rows, cols = n + 1, 2 * n + 2
    j = torch.arange(rows, device="cuda")[:, None]
    i = torch.arange(cols, device="cuda")[None, :]
    x = (i - 0.5) * (dx / 2.0) + 0.0 * j
    y = j * dy + torch.where((i + j) % 2 == 1, -dy / 6.0, dy / 6.0)
    xy = torch.stack([x.double(), y.double()], dim=-1)
    side = min(dx, dy) / 2.0
    xy += _uniform(_generator(seed, 2), -0.1 * side, 0.1 * side, rows, cols, 2)
    r = torch.arange(n, device="cuda")[:, None]
    c = torch.arange(n, device="cuda")[None, :]
    a = 2 * c + r % 2
    lower, upper = r * cols + a, (r + 1) * cols + a
    faces = torch.stack([lower, lower + 1, lower + 2, upper + 2, upper + 1, upper], dim=-1).reshape(-1, 6)
    return xy.reshape(-1, 2).contiguous(), faces.to(torch.int32).contiguous()


def _mesh(kind, cells, shape_seed, seed):
    """A mesh whose geometry is ``shape_seed``'s and whose order of faces is ``seed``'s."""
    if kind == "hexagons":
        v, f = _hexagons(cells, shape_seed)
    elif kind == "triangles":
        v, f = _grid_mesh(cells, 1.0, shape_seed)
    else:
        v, f = _grid_mesh(cells, 1.0 / 3.0, shape_seed)
    return v, _in_order(f, seed, kind == "mixed")


def _shuffled(q, seed):
    return q[torch.randperm(q.shape[0], generator=_generator(seed, 9), device="cuda")]


def _side(kind, cells):
    """The grid spacing behind a mesh of about ``cells`` cells."""
    return LENGTH / math.sqrt(cells / {"triangles": 2.0, "mixed": 4.0 / 3.0, "hexagons": 1.0}[kind])


def _points(n, seed):
    """95 % inside the square, the rest in a frame around it, in no order."""
    g = _generator(seed, 3)
    p = _uniform(g, 0.0, LENGTH, n, 2)
    m = n // 20
    frame = 0.05 * LENGTH
    if m:
        out = _uniform(g, -frame, LENGTH + frame, m, 2)
        axis = torch.arange(m, device="cuda") % 2
        low = torch.arange(m, device="cuda") % 4 < 2
        depth = _uniform(g, 0.0, frame, m)
        out[torch.arange(m, device="cuda"), axis] = torch.where(low, -depth, LENGTH + depth)
        p[torch.randperm(n, generator=g, device="cuda")[:m]] = out
    return p


def _boxes(n, h, seed):
    g = _generator(seed, 4)
    c = _uniform(g, 0.0, LENGTH, n, 2)
    wh = torch.exp(_uniform(g, math.log(BOX_LO * h), math.log(BOX_HI * h), n, 2))
    lo, hi = c - 0.5 * wh, c + 0.5 * wh
    return torch.stack([lo[:, 0], hi[:, 0], lo[:, 1], hi[:, 1]], dim=1).contiguous()


def _segments(n, h, seed):
    g = _generator(seed, 5)
    a = _uniform(g, 0.0, LENGTH, n, 2)
    length = torch.exp(_uniform(g, math.log(SEG_LO * h), math.log(SEG_HI * h), n))
    angle = _uniform(g, 0.0, 2.0 * math.pi, n)
    b = a + torch.stack([length * torch.cos(angle), length * torch.sin(angle)], dim=1)
    return torch.stack([a, b], dim=1).contiguous()


def _batch_sizes(case):
    """(cells, points, segments) of each mesh: even over their logarithms, the three not in step."""
    m = int(case["meshes"])
    out = []
    for k in range(m):
        f = [((k * s) % m + 0.5) / m for s in _strides(m)]
        out.append((int(1e3 * (case["cells"] / 1e3) ** f[0]), int(1e3 * 1e3 ** f[1]), int(1e2 * 1e3 ** f[2])))
    return out


def _strides(m):
    """Three multipliers prime to m, so that k * s mod m runs over all of 0 .. m - 1."""
    found = [s for s in range(1, 8 * m + 16) if math.gcd(s, m) == 1 and (s == 1 or s % m not in (0, 1))]
    return (1, found[min(len(found) - 1, len(found) // 3)], found[min(len(found) - 1, len(found) // 2)])


def _inputs(case, seed):
    """The arrays of a case: the mesh (v, f) and its queries q, target mesh (tv, tf), fields F or output
    gradient G."""
    op, kind, cells = case["op"], case["kind"], case["cells"]
    fixed = op in ("points", "regrid_grad", "barycentric_grad")  # outputs of one shape whatever the geometry
    shape_seed = seed if fixed else 0
    pose = _Pose(seed, turn=op != "build")
    v, f = _mesh(kind, cells, shape_seed, seed)
    out = {"v": pose.xy(v), "f": f}
    h = _side(kind, cells)
    if op in ("points", "barycentric_grad"):
        out["q"] = pose.xy(_points(case["queries"], seed))
    elif op == "boxes":
        out["q"] = pose.boxes(_shuffled(_boxes(case["queries"], h, shape_seed), seed))
    elif op == "segments":
        out["q"] = pose.xy(_shuffled(_segments(case["queries"], h, shape_seed), seed))
    elif op in ("faces", "regrid_setup", "regrid_grad"):
        tv, tf = _mesh("hexagons", case["targets"], shape_seed + 1, seed + 1)
        out["tv"], out["tf"] = pose.xy(tv), tf
    g = _generator(seed, 6)
    if op == "regrid_grad":
        nf = int(case["fields"])
        centre = v[f[:, :3].long()].mean(dim=1)
        waves = _uniform(g, -0.05, 0.05, 2, nf)
        out["F"] = 2.0 + torch.sin(centre @ waves + _uniform(g, 0.0, 2.0 * math.pi, nf))
        out["G"] = torch.randn(tf.shape[0], nf, generator=g, device="cuda", dtype=torch.float64)
    elif op == "barycentric_grad":
        out["G"] = torch.randn(case["queries"], 3, generator=g, device="cuda", dtype=torch.float64)
    return out


def _batch_inputs(case, seed):
    meshes, points, segments = [], [], []
    for k, (cells, n_points, n_segments) in enumerate(_batch_sizes(case)):
        pose = _Pose(int(seed) * 1_009 + k)
        v, f = _mesh(case["kind"], cells, k, int(seed) * 1_009 + k)
        meshes.append((pose.xy(v), f))
        points.append(pose.xy(_points(n_points, int(seed) * 1_009 + k)))
        segments.append(pose.xy(_shuffled(_segments(n_segments, _side(case["kind"], cells), k), int(seed) * 1_009 + k)))
    return meshes, points, segments


# ------------------------------------------------------------------------------------ one pass
def prepare(case, seed):
    op, s = case["op"], {"op": case["op"]}
    if op == "batch":
        meshes, points, segments = _batch_inputs(case, seed)
        batch = TreeBatch([CellTree2d(v, f, -1) for v, f in meshes])
        pts, point_counts = concat_queries(points, 2)
        segs, segment_counts = concat_queries(segments, 4)
        s["graph"] = BatchGraph(batch, pts, point_counts, segs.reshape(-1, 2, 2), segment_counts)
        return s
    a = _inputs(case, seed)
    if op == "build":
        s.update(v=a["v"], f=a["f"], n_buckets=case["n_buckets"], cells_per_leaf=case["cells_per_leaf"])
        return s
    s["tree"] = CellTree2d(a["v"], a["f"], -1)
    if op == "regrid_grad":
        s["regridder"] = Regridder(s["tree"], a["tv"], a["tf"], -1)
        s["F"], s["sv"], s["tv"] = (a[k].requires_grad_() for k in ("F", "v", "tv"))
        s["G"] = a["G"]
    elif op == "barycentric_grad":
        s["v"], s["p"], s["G"] = a["v"].requires_grad_(), a["q"].requires_grad_(), a["G"]
    else:
        s.update({k: a[k] for k in ("q", "tv", "tf") if k in a})
    return s


def run(s):
    op = s["op"]
    if op == "build":
        tree = CellTree2d(s["v"], s["f"], -1, s["n_buckets"], s["cells_per_leaf"])
        return {"nodes": tree.d_nodes, "cells": tree.d_bb_indices, "boxes": tree.d_bb_coords, "depth": tree.depth}
    if op == "points":
        return s["tree"].locate_points(s["q"])
    if op == "boxes":
        return s["tree"].locate_boxes(s["q"])
    if op == "segments":
        return s["tree"].intersect_edges(s["q"])
    if op == "faces":
        return s["tree"].intersect_faces(s["tv"], s["tf"], -1)
    if op == "regrid_setup":
        w = Regridder(s["tree"], s["tv"], s["tf"], -1).weights()
        return w.crow_indices, w.col_indices, w.values
    if op == "regrid_grad":
        y = s["regridder"](s["F"], src_vertices=s["sv"], tgt_vertices=s["tv"])
        return (y.detach(),) + torch.autograd.grad(y, (s["F"], s["sv"], s["tv"]), s["G"])
    if op == "barycentric_grad":
        face, w = barycentric_weights(s["tree"], s["p"], s["v"])
        return (face, w.detach()) + torch.autograd.grad(w, (s["p"], s["v"]), s["G"])
    s["graph"].replay()
    r = s["graph"].result()
    return r.cells, r.ii, r.jj, r.xy


# ------------------------------------------------------------------------------------ what a pass needs
def _mesh_bytes(kind, cells):
    """Vertices (two doubles) and int32 face rows of a mesh."""
    vertices, width = {"triangles": (0.5, 3), "mixed": (0.75, 4), "hexagons": (2.0, 6)}[kind]
    return cells * (16.0 * vertices + 4.0 * width)


def _cell_perimeter(kind, h):
    """The mean perimeter of a cell of a mesh with grid spacing h."""
    return {"triangles": (2.0 + math.sqrt(2.0)) * h, "mixed": 0.5 * (4.0 + 2.0 + math.sqrt(2.0)) * h,
            "hexagons": math.sqrt(8.0 * math.sqrt(3.0)) * h}[kind]


def _box_hits(kind):
    """Cells whose boxes meet a query box, on average: density x mean of (w + c) (h + c), c the mean
    width of a cell's box."""
    mean = (BOX_HI - BOX_LO) / math.log(BOX_HI / BOX_LO)
    density, c = {"triangles": (2.0, 1.12), "mixed": (4.0 / 3.0, 1.12), "hexagons": (1.0, 1.2)}[kind]
    return density * (mean + c) ** 2


def _segment_hits(kind):
    """Cells a segment passes: 1 + length x edge length per area x 2 / pi."""
    mean = (SEG_HI - SEG_LO) / math.log(SEG_HI / SEG_LO)
    cells_per_area = {"triangles": 2.0, "mixed": 4.0 / 3.0, "hexagons": 1.0}[kind]
    return 1.0 + mean * 0.5 * cells_per_area * _cell_perimeter(kind, 1.0) * 2.0 / math.pi


def _overlaps(case):
    """Overlapping pairs of two convex meshes over one square: n_s + n_t + the mean number of crossings."""
    ns, nt = case["cells"], case["targets"]
    ps = _cell_perimeter(case["kind"], _side(case["kind"], ns))
    pt = _cell_perimeter("hexagons", _side("hexagons", nt))
    return ns + nt + ps * pt * ns * nt / (2.0 * math.pi * LENGTH * LENGTH)


CLIP_FLOPS = 212.0      # Sutherland-Hodgman and area of a kept pair (counted in tests/golden/flops_overlap.json)
SAT_FLOPS = 297.0       # separating axes of a pair, likewise
ADJOINT_FLOPS = 620.0   # derivative of a pair's area in both polygons, likewise
WALK_FLOPS = 60.0       # comparisons and products of one point's cell test


def work(case):
    op, kind, cells = case["op"], case["kind"], float(case["cells"])
    mesh = _mesh_bytes(kind, cells)
    tree = 32.0 * 1.2 * cells + 4.0 * cells
    if op == "build":
        # the mesh in; nodes, order and boxes out
        return {"bytes": mesh + tree + 32.0 * cells, "flops": 10.0 * cells}
    if op == "batch":
        total = {"bytes": 0.0, "flops": 0.0}
        for c, p, e in _batch_sizes(case):
            rows = e * _segment_hits(kind)
            total["bytes"] += min(_mesh_bytes(kind, c) + 42.4 * c, 150.0 * (p + rows)) + 24.0 * p + 32.0 * e + 48.0 * rows
            total["flops"] += WALK_FLOPS * p + 80.0 * rows
        return total
    if op in ("points", "barycentric_grad"):
        n = float(case["queries"])
        out = 8.0 if op == "points" else 8.0 + 24.0 + 24.0 + 16.0
        more = 0.0 if op == "points" else 16.0 * 0.5 * cells
        return {"bytes": n * (16.0 + out) + min(mesh + tree, 150.0 * n) + more,
                "flops": n * (WALK_FLOPS if op == "points" else WALK_FLOPS + 120.0)}
    if op == "boxes":
        n = float(case["queries"])
        rows = n * _box_hits(kind)
        return {"bytes": 32.0 * n + 16.0 * rows + min(tree + 32.0 * cells, 100.0 * rows), "flops": 4.0 * rows}
    if op == "segments":
        n = float(case["queries"])
        rows = n * _segment_hits(kind)
        return {"bytes": 32.0 * n + 48.0 * rows + min(mesh + tree + 32.0 * cells, 150.0 * rows), "flops": 80.0 * rows}
    pairs = _overlaps(case)
    both = mesh + _mesh_bytes("hexagons", float(case["targets"]))
    if op == "faces":
        return {"bytes": both + tree + 24.0 * pairs, "flops": (SAT_FLOPS + CLIP_FLOPS) * pairs}
    if op == "regrid_setup":
        return {"bytes": both + tree + 16.0 * pairs + 8.0 * case["targets"], "flops": (SAT_FLOPS + CLIP_FLOPS) * pairs}
    nf, nt = float(case["fields"]), float(case["targets"])
    # pairs, both meshes, F and G in; y, dF and the vertex gradients out
    return {"bytes": 8.0 * pairs + 2.0 * both + 16.0 * nf * (cells + nt),
            "flops": pairs * (CLIP_FLOPS + ADJOINT_FLOPS + 6.0 * nf)}


# ------------------------------------------------------------------------------------ 64-bit values
def _rows(v, f):
    """(n, k, 2) corner coordinates, rows shorter than k padded by their last vertex."""
    f = f.long()
    for k in range(3, f.shape[1]):
        f = torch.cat([f[:, :k], torch.where(f[:, k:k + 1] < 0, f[:, k - 1:k], f[:, k:k + 1]), f[:, k + 1:]], dim=1)
    return f, v[f]


def _face_boxes(v, f):
    _, c = _rows(v, f)
    lo, hi = c.amin(dim=1), c.amax(dim=1)
    return torch.stack([lo[:, 0], hi[:, 0], lo[:, 1], hi[:, 1]], dim=1)


def _spread(starts, counts):
    """(owner, value) of the ranges [starts, starts + counts), one after the other."""
    owner = torch.repeat_interleave(torch.arange(counts.numel(), device=counts.device), counts)
    first = torch.cumsum(counts, 0) - counts
    return owner, starts[owner] + torch.arange(owner.numel(), device=counts.device) - first[owner]


class _Bins:
    """Boxes in square bins by their lower corner, for finding the boxes near a query box."""

    def __init__(self, boxes):
        self.x0, self.y0 = float(boxes[:, 0].min()), float(boxes[:, 2].min())
        self.b = float(torch.maximum(boxes[:, 1] - boxes[:, 0], boxes[:, 3] - boxes[:, 2]).max()) * 1.0000001
        bx, by = self.bin(boxes[:, 0], self.x0), self.bin(boxes[:, 2], self.y0)
        self.nx, self.ny = int(bx.max()) + 1, int(by.max()) + 1
        key = by * self.nx + bx
        self.ids = torch.argsort(key, stable=True)
        count = torch.bincount(key, minlength=self.nx * self.ny)
        self.start = torch.cat([count.new_zeros(1), torch.cumsum(count, 0)])

    def bin(self, x, x0):
        return torch.floor((x - x0) / self.b).long()

    def near(self, q):
        """(query, box) of all boxes that may meet the query boxes (xmin, xmax, ymin, ymax)."""
        x0 = (self.bin(q[:, 0], self.x0) - 1).clamp(0, self.nx)
        x1 = (self.bin(q[:, 1], self.x0) + 1).clamp(0, self.nx)
        y0 = (self.bin(q[:, 2], self.y0) - 1).clamp(0, self.ny)
        y1 = (self.bin(q[:, 3], self.y0) + 1).clamp(0, self.ny)
        owner, row = _spread(y0, (y1 - y0).clamp(min=0))
        lo = self.start[row * self.nx + x0[owner]]
        hi = self.start[row * self.nx + torch.maximum(x1, x0)[owner]]
        part, at = _spread(lo, hi - lo)
        return owner[part], self.ids[at]


def _cross(u, v):
    return u[..., 0] * v[..., 1] - u[..., 1] * v[..., 0]


def _clip_range(a, d, poly, closed):
    """(t0, t1): where a + t d, t in [0, 1], lies in the counter-clockwise polygons (leading dimensions
    of a broadcast against poly's)."""
    e = torch.roll(poly, -1, dims=-2) - poly
    num = _cross(e, a.unsqueeze(-2) - poly)      # > 0: a is inside this edge's line
    den = _cross(e, d.unsqueeze(-2).expand_as(e))
    flat = den == 0.0
    t = -num / torch.where(flat, torch.ones_like(den), den)
    real = (e != 0.0).any(dim=-1)
    out = flat & real & ((num < 0.0) if closed else (num <= 0.0))
    t0 = torch.where(~flat & (den > 0.0), t, torch.zeros_like(t)).amax(dim=-1).clamp(min=0.0)
    t1 = torch.where(~flat & (den < 0.0), t, torch.ones_like(t)).amin(dim=-1).clamp(max=1.0)
    return t0, torch.where(out.any(dim=-1), t0, t1)


def _clipped_segments(v, f, segs, chunk=50_000):
    """(rows, 2, 2): the pieces of every segment in every face, by segment and along it."""
    _, corners = _rows(v, f)
    bins = _Bins(_face_boxes(v, f))
    out = []
    for k in range(0, segs.shape[0], chunk):
        s = segs[k:k + chunk]
        lo, hi = s.amin(dim=1), s.amax(dim=1)
        q, c = bins.near(torch.stack([lo[:, 0], hi[:, 0], lo[:, 1], hi[:, 1]], dim=1))
        a, d = s[q, 0], s[q, 1] - s[q, 0]
        side = _cross(d.unsqueeze(1), corners[c] - a.unsqueeze(1))
        touch = (side.amin(dim=1) < 0.0) & (side.amax(dim=1) > 0.0)
        q, c, a, d = q[touch], c[touch], a[touch], d[touch]
        t0, t1 = _clip_range(a, d, corners[c], True)
        hit = t1 > t0
        q, a, d, t0, t1 = q[hit], a[hit], d[hit], t0[hit], t1[hit]
        order = torch.argsort(q.double() * 2.0 + t0)
        piece = torch.stack([a + t0[:, None] * d, torch.where((t1 == 1.0)[:, None], s[q, 1], a + t1[:, None] * d)], dim=1)
        out.append(piece[order])
    return torch.cat(out)


def _polygon_area(p):
    return 0.5 * _cross(p - p[..., :1, :], torch.roll(p, -1, dims=-2) - p[..., :1, :]).sum(dim=-1)


def _overlap_area(p, q):
    """Area of the intersections of counter-clockwise convex polygons p (n, j, 2) and q (n, k, 2): half
    the boundary integral over the pieces of either polygon's edges that lie in the other."""
    o = p[:, :1].detach()
    p, q = p - o, q - o
    total = p.new_zeros(p.shape[0])
    for u, w, closed in ((p, q, True), (q, p, False)):
        d = torch.roll(u, -1, dims=1) - u
        t0, t1 = _clip_range(u, d, w.unsqueeze(1).expand(-1, u.shape[1], -1, -1), closed)
        total = total + ((t1 - t0).clamp(min=0.0) * _cross(u, d)).sum(dim=1)
    return 0.5 * total


def _exact_regrid(case, seed, chunk=200_000):
    a = _inputs(case, seed)
    sv, sf, tv, tf, F, G = (a[k] for k in ("v", "f", "tv", "tf", "F", "G"))
    sv.requires_grad_(), tv.requires_grad_()
    si, _ = _rows(sv.detach(), sf)
    ti = tf.long()
    bins = _Bins(_face_boxes(sv.detach(), sf))
    tb = _face_boxes(tv.detach(), tf)
    area = _polygon_area(tv.detach()[ti])
    y, gF = torch.zeros_like(G), torch.zeros_like(F)
    step = max(1, chunk // max(4, int(4.0 * case["cells"] / case["targets"])))
    for k in range(0, tf.shape[0], step):
        t, s = bins.near(tb[k:k + step])
        t = t + k
        with torch.no_grad():
            over = _overlap_area(tv[ti[t]], sv[si[s]])
        t, s = t[over > 0.0], s[over > 0.0]
        A = _overlap_area(tv[ti[t]], sv[si[s]])
        share = (A.detach() / area[t])[:, None]
        y.index_add_(0, t, share * F[s])
        gF.index_add_(0, s, share * G[t])
        ((G[t] * F[s]).sum(dim=1) / area[t] * A).sum().backward()
    (-((G * y).sum(dim=1) / area) * _polygon_area(tv[ti])).sum().backward()
    return y, gF, sv.grad, tv.grad


def _exact_barycentric(case, seed, chunk=200_000):
    a = _inputs(case, seed)
    v, f, p, G = a["v"], a["f"].long(), a["q"], a["G"]
    bins = _Bins(_face_boxes(v, f))
    face = torch.full((p.shape[0],), -1, dtype=torch.long, device=p.device)
    for k in range(0, p.shape[0], chunk):
        c = p[k:k + chunk]
        q, t = bins.near(torch.stack([c[:, 0], c[:, 0], c[:, 1], c[:, 1]], dim=1))
        w = v[f[t]]
        inside = (_cross(torch.roll(w, -1, dims=1) - w, c[q].unsqueeze(1) - w) >= 0.0).all(dim=1)
        face[k + q[inside]] = t[inside]
    p.requires_grad_(), v.requires_grad_()
    m = face >= 0
    a, b, c = v[f[face[m]]].unbind(dim=1)
    area = _cross(b - a, c - a).abs()
    w2 = _cross(b - a, p[m] - a).abs() / area
    w1 = _cross(c - a, p[m] - a).abs() / area
    w = p.new_zeros(p.shape[0], 3).index_put((torch.nonzero(m)[:, 0],), torch.stack([1.0 - w1 - w2, w1, w2], dim=1))
    gp, gv = torch.autograd.grad(w, (p, v), G)
    return None, w.detach(), gp, gv


def exact(case, seed):
    op = case["op"]
    if op == "build":
        a = _inputs(case, seed)
        return {"nodes": None, "cells": None, "boxes": _face_boxes(a["v"], a["f"]), "depth": None}
    if op == "segments":
        a = _inputs(case, seed)
        return None, None, _clipped_segments(a["v"], a["f"], a["q"])
    if op == "batch":
        meshes, _, segments = _batch_inputs(case, seed)
        return None, None, None, torch.cat([_clipped_segments(v, f, s) for (v, f), s in zip(meshes, segments)])
    if op == "regrid_grad":
        return _exact_regrid(case, seed)
    if op == "barycentric_grad":
        return _exact_barycentric(case, seed)
    return None
