"""Intersection, get_intersection and dual_contouring -- drop-ins for the
reference's DC front end and solver.

Reference: Intersection (include/its.cuh:6-26, bound at
src/isoext_ext.cu:305-327), get_intersection (src/its.cu:93-159, bound at
src/isoext_ext.cu:329-343), dual_contouring (src/dc.cu:161-218, bound at
src/isoext_ext.cu:345-378 with its default-normals logic).

Differences on purpose:
* get_points()/get_normals() return copies; the reference hands over its
  buffer on the first call and leaves the object empty
  (src/isoext_ext.cu:67-76).
* Quads whose four cells do not all exist are skipped; the reference indexes
  past the grid's upper faces (include/utils.cuh:130-134).
* The QEF is solved per cell in FP32 centred at the mass point and scaled by
  the cell size, refined once, and re-solved in FP64 exactly as the
  reference poses it when the condition number exceeds min(1e6, 0.5/svd_tol).
* Vertex order is active-cell order (the reference sorts positions); faces
  keep the reference's quad order.
"""

from __future__ import annotations

import ctypes
import threading

import torch

from . import _lib, workspace
from .grid import check_cuda_f32

P = ctypes.POINTER


class IsoGrid(ctypes.Structure):
    _fields_ = [("values", ctypes.c_void_p), ("sparse_cell_ids", ctypes.c_void_p), ("n_sparse", ctypes.c_int64),
                ("shape", ctypes.c_int64 * 3), ("aabb_min", ctypes.c_float * 3), ("aabb_max", ctypes.c_float * 3)]


class IsoIts(ctypes.Structure):
    _fields_ = [("ncells", ctypes.c_int64), ("npts", ctypes.c_int64), ("cell_indices", ctypes.c_void_p),
                ("cell_dense", ctypes.c_void_p), ("cell_offsets", ctypes.c_void_p), ("points", ctypes.c_void_p),
                ("normals", ctypes.c_void_p), ("edge_local", ctypes.c_void_p), ("is_out", ctypes.c_void_p),
                ("entry_cell", ctypes.c_void_p), ("amask_tab", ctypes.c_void_p), ("apre_tab", ctypes.c_void_p)]


vp, i64, f32 = ctypes.c_void_p, ctypes.c_int64, ctypes.c_float
_lib.declare("isoext_its_scratch_bytes", i64, [P(IsoGrid)])
_lib.declare("isoext_its_count", ctypes.c_int, [P(IsoGrid), f32, vp, i64, i64 * 2, vp])
_lib.declare("isoext_its_table_entries", i64, [i64 * 3])
_lib.declare("isoext_its_emit", ctypes.c_int, [P(IsoGrid), f32, vp, i64, i64, vp, vp, vp, vp, vp, vp, vp, vp, vp, vp,
                                               vp])
_lib.declare("isoext_its_begin", ctypes.c_int, [P(IsoGrid), f32, vp, i64, vp])
_lib.declare("isoext_its_finish", ctypes.c_int, [P(IsoGrid), f32, vp, i64, i64, vp, vp, vp, vp, vp, vp, vp, vp, vp, vp,
                                                 i64 * 2, vp])
_lib.declare("isoext_dc_grid_workspace_bytes", i64, [P(IsoGrid), i64])
_lib.declare("isoext_dc_grid", ctypes.c_int, [P(IsoGrid), f32, f32, f32, vp, i64, i64, vp, i64, vp, i64, i64 * 5, vp])
_lib.declare("isoext_its_normals", ctypes.c_int, [P(IsoGrid), P(IsoIts), vp, vp])
_lib.declare("isoext_dc_workspace_bytes", i64, [i64, i64])
_lib.declare("isoext_dc", ctypes.c_int, [P(IsoGrid), P(IsoIts), f32, f32, vp, i64, vp, i64, vp, i64, vp, vp,
                                         _lib.I64x4, vp])
_lib.declare("isoext_dc_backward", ctypes.c_int, [P(IsoGrid), P(IsoIts), f32, f32, f32, i64, vp, vp, vp, vp, vp])
_lib.declare("isoext_mc_sparse_count", ctypes.c_int, [P(IsoGrid), f32, vp, P(i64), vp])
_lib.declare("isoext_mc_sparse", ctypes.c_int, [P(IsoGrid), f32, ctypes.c_int, i64, vp, i64, vp, i64, vp, i64, vp,
                                                i64 * 2, vp])


def grid_struct(grid) -> IsoGrid:
    g = IsoGrid()
    g.values = grid.values.data_ptr() if grid.values.numel() else None
    ids = getattr(grid, "cell_ids", None)
    if ids is not None:
        g.sparse_cell_ids = ids.data_ptr() if ids.numel() else None
        g.n_sparse = ids.numel()
    else:
        g.sparse_cell_ids = None
        g.n_sparse = 0
    for i in range(3):
        g.shape[i] = int(grid.shape[i])
        g.aabb_min[i] = float(grid.aabb_min[i])
        g.aabb_max[i] = float(grid.aabb_max[i])
    return g


class Intersection:
    """Edge/surface intersections of a grid (points, optional normals)."""

    def __init__(self, grid, level, cell_indices, cell_dense, cell_offsets, points, normals, edge_local, is_out,
                 entry_cell, tables=None):
        self._grid = grid
        self._level = float(level)
        self.cell_indices = cell_indices
        self.cell_dense = cell_dense
        self.cell_offsets = cell_offsets
        self.points = points
        self.normals = normals if normals is not None else torch.zeros_like(points)
        self.edge_local = edge_local
        self.is_out = is_out
        self.entry_cell = entry_cell
        # dense grids: per (cell row, 64-cell word) active masks and first
        # active indices, the neighbour lookups of dual contouring's quads
        self._tables = tables
        self._has_normals = normals is not None

    def get_points(self) -> torch.Tensor:
        """(N, 3) float32 intersection points (a copy)."""
        return self.points.clone()

    def get_normals(self) -> torch.Tensor:
        """(N, 3) float32 normals (a copy; zeros until set or computed)."""
        return self.normals.clone()

    def has_normals(self) -> bool:
        return self._has_normals

    def set_normals(self, new_normals: torch.Tensor) -> None:
        """Copy (N, 3) float32 normals in (src/isoext_ext.cu:318-327)."""
        check_cuda_f32(new_normals, ndim=2, last=3, name="new_normals")
        if new_normals.shape != self.points.shape:
            raise RuntimeError("Cannot set values with different shapes")
        self.normals = new_normals.detach().clone()
        self._has_normals = True

    def __len__(self):
        return self.points.shape[0]

    def _struct(self, normals=None, grid=None) -> IsoIts:
        s = IsoIts()
        s.ncells = self.cell_indices.numel()
        s.npts = self.points.shape[0]
        s.cell_indices = self.cell_indices.data_ptr()
        s.cell_dense = self.cell_dense.data_ptr()
        s.cell_offsets = self.cell_offsets.data_ptr()
        s.points = self.points.data_ptr()
        n = self.normals if normals is None else normals
        s.normals = n.data_ptr()
        s.edge_local = self.edge_local.data_ptr()
        s.is_out = self.is_out.data_ptr()
        s.entry_cell = self.entry_cell.data_ptr()
        # the tables index cell rows of the grid shape they were built for
        same_shape = grid is None or [int(x) for x in grid.shape] == [int(x) for x in self._grid.shape]
        if self._tables is not None and same_shape and getattr(grid, "cell_ids", None) is None:
            s.amask_tab = self._tables[0].data_ptr()
            s.apre_tab = self._tables[1].data_ptr()
        return s


def _device(grid):
    return grid.values.device


def get_intersection(grid, level: float = 0.0, compute_normals: bool = False) -> Intersection:
    """Crossing-edge intersection points of the grid at `level`
    (linear interpolation, src/its.cu:37-90); with compute_normals, trilinear
    central-difference normals (src/its.cu:186-268)."""
    dev = _device(grid)
    L = _lib.lib()
    g = grid_struct(grid)
    nbytes = L.isoext_its_scratch_bytes(ctypes.byref(g)) if g.values else 64
    scratch = workspace.get("its", nbytes, dev)
    counts = (ctypes.c_int64 * 2)()
    tables = None
    with torch.cuda.device(dev):
        stream = _lib.stream_ptr(dev)
        shape = tuple(g.shape)
        dense = getattr(grid, "cell_ids", None) is None
        if dense:
            nt = max(int(L.isoext_its_table_entries(g.shape)), 1)
        if dense and not _its_vary(shape):
            # the buffers, sized by recent sets of this shape, are made while the count runs, and only the counts are
            # waited for
            _lib.check(L.isoext_its_begin(ctypes.byref(g), float(level), scratch.data_ptr(), scratch.numel(), stream),
                       "get_intersection")
            tables = (torch.empty(nt, dtype=torch.int64, device=dev), torch.empty(nt, dtype=torch.int32, device=dev))
            nc, npt = _its_caps(shape)
            for _ in range(2):
                b = _its_buffers(nc, npt, compute_normals, dev)
                rc = L.isoext_its_finish(ctypes.byref(g), float(level), scratch.data_ptr(), nc, npt,
                                         *(t.data_ptr() if t is not None else None for t in b), tables[0].data_ptr(),
                                         tables[1].data_ptr(), counts, stream)
                if rc != _lib.E_CAPACITY:
                    break
                nc, npt = int(counts[0]), int(counts[1])
            _lib.check(rc, "get_intersection")
            cap, nc, npt = npt, int(counts[0]), int(counts[1])
            ends = (nc, nc, nc + 1, npt, npt, npt, npt, npt)
            b = [t[:n] if t is not None else None for t, n in zip(b, ends)]
            if cap > 2 * npt + _PINNED:   # do not pin much larger buffers behind a small set
                b = [t.clone() if t is not None else None for t in b]
        elif not dense and g.n_sparse == 0:
            b = _its_buffers(0, 0, compute_normals, dev)
            b[2].zero_()
        else:
            _lib.check(L.isoext_its_count(ctypes.byref(g), float(level), scratch.data_ptr(), scratch.numel(), counts,
                                          stream), "get_intersection")
            nc, npt = int(counts[0]), int(counts[1])
            b = _its_buffers(nc, npt, compute_normals, dev)
            if dense:
                tables = (torch.empty(nt, dtype=torch.int64, device=dev),
                          torch.empty(nt, dtype=torch.int32, device=dev))
            p = [t.data_ptr() if t is not None and (npt or k < 3) else None for k, t in enumerate(b)]
            _lib.check(L.isoext_its_emit(ctypes.byref(g), float(level), scratch.data_ptr(), nc, npt, *p,
                                         *(t.data_ptr() for t in tables or ()), *(() if dense else (None, None)),
                                         stream), "get_intersection")
        if dense:
            _remember(_its_hint, shape, (nc, npt), _its_low)
            tables = tables if nc else None
    cell_indices, cell_dense, cell_offsets, points, normals, edge_local, is_out, entry_cell = b
    return Intersection(grid, level, cell_indices, cell_dense, cell_offsets, points, normals, edge_local, is_out,
                        entry_cell, tables)


# cells and points of a dense shape's recent intersection sets, and cells,
# vertices and faces of its recent dual meshes (sizing hints); points of its
# recent small intersection sets
_its_hint: dict = {}
_dc_hint: dict = {}
_its_low: dict = {}
# dense shapes whose last dual mesh had no cell: often the next has none either
# (blocks of a larger grid), and a call that only counts takes 39 us where the
# whole one takes 73 (128^3)
_dc_none: set = set()
_hint_lock = threading.Lock()
_PINNED = 65536   # entries that may be kept behind a smaller set, beyond its own size


def _remember(hints, shape, sizes, low=None):
    """The sizes of a call, or what is left of larger ones before it: those
    fall by a 32nd a call.  With the eighth more that the next call makes room
    for, a large surface still fits after three small ones of its shape (too
    little room costs a second run), and a lone large one is soon forgotten.
    low: the last size from the other side, an eighth of the way a call."""
    if hints.get(shape) == sizes and (low is None or low.get(shape) == sizes[-1]):
        return   # nothing changes: no lock
    with _hint_lock:
        if len(hints) > 4096:
            hints.clear()
        hints[shape] = tuple([max(n, o - o // 32) for n, o in zip(sizes, hints.get(shape, sizes))])
        if low is not None:
            if len(low) > 4096:
                low.clear()
            o = low.get(shape, sizes[-1])
            low[shape] = min(sizes[-1], o + (sizes[-1] - o + 7) // 8)


def _its_vary(shape):
    """Whether a shape's recent intersection sets differ so much that room for
    the largest would mean copying the others out of it (eight copies, 40 us,
    where waiting for the count before the buffers are made takes 20)."""
    hint, low = _its_hint.get(shape), _its_low.get(shape)
    return hint is not None and low is not None and hint[1] + (hint[1] >> 3) + 4096 > 2 * low + _PINNED


# Most cells that a call without a hint makes room for; a call that needs more
# is repeated with the counted size.
_FIRST_CELLS = 1 << 22


def _most_cells(shape):
    X, Y, Z = shape
    return (X - 1) * (Y - 1) * (Z - 1) if X > 1 and Y > 1 and Z > 1 else 1


def _first_cells(shape):
    # surface-like: a few times the largest cross-section
    X, Y, Z = shape
    return min(max(1 << 15, 2 * max(X * Y, Y * Z, X * Z)), _FIRST_CELLS, _most_cells(shape))


def _its_caps(shape):
    hint = _its_hint.get(shape)   # a single dict read needs no lock
    if hint is None:
        cells = _first_cells(shape)
        return cells, 4 * cells
    c, p = hint
    most = min(_most_cells(shape), 0x7fffffff)
    return min(c + (c >> 3) + 1024, most), min(p + (p >> 3) + 4096, 12 * most)


def _dc_caps(shape):
    hint = _dc_hint.get(shape)
    if hint is None:
        nc = _first_cells(shape)
        return nc, nc, 2 * nc
    c, v, f = hint
    most = min(_most_cells(shape), 0x3fffffff)
    return min(c + (c >> 3) + 1024, most), min(v + (v >> 3) + 1024, most), min(f + (f >> 3) + 1024, 6 * most)


def _its_buffers(nc, npt, normals, dev):
    """Cell indices, dense ids, offsets, points, normals, local edges, orientations, entry cells."""
    i64t, f32t, u8t = (dict(dtype=t, device=dev) for t in (torch.int64, torch.float32, torch.uint8))
    return [torch.empty(nc, **i64t), torch.empty(nc, **i64t), torch.empty(nc + 1, **i64t),
            torch.empty((npt, 3), **f32t), torch.empty((npt, 3), **f32t) if normals else None, torch.empty(npt, **u8t),
            torch.empty(npt, **u8t), torch.empty(npt, dtype=torch.int32, device=dev)]


def compute_normals(grid, its: Intersection) -> torch.Tensor:
    """Trilinear central-difference normals for an intersection set."""
    dev = _device(grid)
    out = torch.empty_like(its.points)
    if its.points.shape[0] == 0:
        return out
    g = grid_struct(grid)
    s = its._struct(normals=out)
    with torch.cuda.device(dev):
        _lib.check(_lib.lib().isoext_its_normals(ctypes.byref(g), ctypes.byref(s), out.data_ptr(),
                                                 _lib.stream_ptr(dev)), "compute normals")
    return out


def dc_raw(grid, its: Intersection, normals: torch.Tensor, reg: float, svd_tol: float, want_dual: bool = False,
           want_vcell: bool = False):
    """Run the DC kernels; returns (v, f, info[, dual_v]); with want_vcell,
    info["vcell"] holds the active cell of each output vertex."""
    dev = _device(grid)
    L = _lib.lib()
    g = grid_struct(grid)
    s = its._struct(normals=normals, grid=grid)
    nc, npt = int(s.ncells), int(s.npts)
    ws = workspace.get("dc", L.isoext_dc_workspace_bytes(nc, npt), dev)
    out_v = torch.empty((max(nc, 1), 3), dtype=torch.float32, device=dev)
    out_f = torch.empty((max(2 * npt, 1), 3), dtype=torch.int32, device=dev)
    dual = torch.empty((max(nc, 1), 3), dtype=torch.float32, device=dev) if want_dual else None
    vcell = torch.empty(max(nc, 1), dtype=torch.int32, device=dev) if want_vcell else None
    counts = _lib.I64x4()
    with torch.cuda.device(dev):
        _lib.check(L.isoext_dc(ctypes.byref(g), ctypes.byref(s), float(reg), float(svd_tol), ws.data_ptr(),
                               ws.numel(), out_v.data_ptr(), out_v.shape[0], out_f.data_ptr(), out_f.shape[0],
                               dual.data_ptr() if dual is not None else None,
                               vcell.data_ptr() if vcell is not None else None, counts, _lib.stream_ptr(dev)),
                   "dual_contouring")
    nv, nf = int(counts[0]), int(counts[1])
    info = {"fp64_resolves": int(counts[2]), "quads": int(counts[3])}
    if want_vcell:
        info["vcell"] = vcell[:nv]
    v, f = out_v[:nv], out_f[:nf]
    if out_v.shape[0] > 2 * nv + 65536:
        v = v.clone()
    if out_f.shape[0] > 2 * nf + 65536:
        f = f.clone()
    if want_dual:
        return v, f, info, dual[:nc]
    return v, f, info


def dual_contouring(grid, level: float = 0.0, intersection: Intersection | None = None, reg: float = 1e-2,
                    svd_tol: float = 1e-6):
    """Extract an iso-surface with Dual Contouring.

    Without `intersection`, intersections and normals are computed at
    `level`; an intersection without normals gets trilinear normals.
    Returns (vertices (N, 3) float32, faces (M, 3) int32) or (None, None).

    On a UniformGrid without `intersection` no intersection set is stored:
    each active cell's crossing edges, points and trilinear normals are
    recomputed from its corner values (the same floats, in the same order, as
    get_intersection(grid, level, True) holds), which gives the same mesh.
    """
    from .grid import UniformGrid
    if intersection is None and isinstance(grid, UniformGrid):
        return _dc_grid(grid, level, reg, svd_tol)
    its = intersection if intersection is not None else get_intersection(grid, level, True)
    if its.points.shape[0] == 0:
        return None, None
    normals = its.normals if its.has_normals() else compute_normals(grid, its)
    v, f, _ = dc_raw(grid, its, normals.contiguous(), reg, svd_tol)
    if f.shape[0] == 0:
        return None, None
    return v, f


def _dc_grid(grid, level: float, reg: float, svd_tol: float):
    """dual_contouring of a dense grid without an intersection set, into
    buffers sized by recent meshes of this shape (one synchronisation)."""
    check_cuda_f32(grid.values, 3, name="values")
    dev = _device(grid)
    L = _lib.lib()
    g = grid_struct(grid)
    shape = tuple(g.shape)
    counts = (ctypes.c_int64 * 5)()
    with torch.cuda.device(dev):
        stream = _lib.stream_ptr(dev)
        if shape in _dc_none:   # the last one of this shape had no cell: look before everything is launched
            few = (ctypes.c_int64 * 2)()
            ws = workspace.get("dc_grid", L.isoext_its_scratch_bytes(ctypes.byref(g)), dev, stream)
            _lib.check(L.isoext_its_count(ctypes.byref(g), float(level), ws.data_ptr(), ws.numel(), few, stream),
                       "dual_contouring")
            if few[0] == 0:
                return None, None
        nc, cap_v, cap_f = _dc_caps(shape)
        for _ in range(3):
            ws = workspace.get("dc_grid", L.isoext_dc_grid_workspace_bytes(ctypes.byref(g), nc), dev, stream)
            out_v = torch.empty((cap_v, 3), dtype=torch.float32, device=dev)
            out_f = torch.empty((cap_f, 3), dtype=torch.int32, device=dev)
            rc = L.isoext_dc_grid(ctypes.byref(g), float(level), float(reg), float(svd_tol), ws.data_ptr(), ws.numel(),
                                  nc, out_v.data_ptr(), cap_v, out_f.data_ptr(), cap_f, counts, stream)
            if rc != _lib.E_CAPACITY:
                break
            if counts[3] > nc:   # cells did not fit: a vertex each at most, and a quad per canonical edge, about as many
                nc = int(counts[3])
                cap_v, cap_f = nc, max(cap_f, 2 * nc)
            else:
                cap_v, cap_f = max(cap_v, int(counts[0])), max(cap_f, int(counts[1]))
    _lib.check(rc, "dual_contouring")
    nv, nf, _, cells, _ = counts
    _remember(_dc_hint, shape, (cells, nv, nf))
    if (shape in _dc_none) != (cells == 0):
        with _hint_lock:
            if len(_dc_none) > 4096:
                _dc_none.clear()
            (_dc_none.discard if cells else _dc_none.add)(shape)
    if nf == 0:
        return None, None
    v, f = out_v[:nv], out_f[:nf]
    if cap_v > 2 * nv + 65536:   # do not pin a much larger allocation behind a small mesh
        v = v.clone()
    if cap_f > 2 * nf + 65536:
        f = f.clone()
    return v, f
