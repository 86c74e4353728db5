"""Ragged batches of dense marching-cubes and dual-contouring extractions.

``mc_batch(jobs)`` extracts every grid of a list of (values, level, method,
aabb) jobs with one launch per stage for the whole batch (classify, count,
scan, emit, special-list gather), in two phases with a single host
synchronisation each: phase 1 sizes every mesh, the outputs are allocated,
phase 2 writes them, then the weld fix-up runs for the grids that need it.
The kernels walk batch-wide index spaces (words, count blocks, tiles) and
find their grid by binary search over a descriptor array uploaded from
pinned memory.  Results are identical to one ``marching_cubes`` call per
grid (tests/test_batch_gpu.py).

``dc_batch(jobs)`` does the same for dual contouring: phase 1 counts every
grid's active cells and intersections (the mask pipeline in intersection
mode), phase 2 writes the concatenated intersection sets with normals and
runs the QEF solve, quad emission and vertex weld of all grids at once; the
meshes come back as views of two shared output buffers.  Results are
identical to ``dual_contouring(grid, level)`` per grid.
"""

from __future__ import annotations

import ctypes
import threading
from dataclasses import dataclass

import torch

from . import _lib, workspace


class McItem(ctypes.Structure):
    _fields_ = [("values", ctypes.c_void_p), ("shape", ctypes.c_int64 * 3), ("aabb_min", ctypes.c_float * 3),
                ("aabb_max", ctypes.c_float * 3), ("level", ctypes.c_float), ("method", ctypes.c_int),
                ("out_v", ctypes.c_void_p), ("cap_v", ctypes.c_int64), ("out_f", ctypes.c_void_p),
                ("cap_f", ctypes.c_int64), ("sdf", ctypes.c_void_p), ("sdf_normals", ctypes.c_int)]


_declared = False
_decl_lock = threading.Lock()


def _decl():
    global _declared
    with _decl_lock:
        if _declared:
            return _lib.lib()
        L = _lib.lib()
        vp, i64, c_int = ctypes.c_void_p, ctypes.c_int64, ctypes.c_int
        L.isoext_mc_batch_workspace_bytes.restype = i64
        L.isoext_mc_batch_workspace_bytes.argtypes = [c_int, ctypes.POINTER(McItem), c_int, i64]
        L.isoext_mc_batch_count.restype = c_int
        L.isoext_mc_batch_count.argtypes = [c_int, ctypes.POINTER(McItem), c_int, vp, i64, i64,
                                            ctypes.POINTER(i64), vp]
        L.isoext_mc_batch_emit.restype = c_int
        L.isoext_mc_batch_emit.argtypes = [c_int, ctypes.POINTER(McItem), c_int, vp, i64, i64,
                                           ctypes.POINTER(i64), vp]
        L.isoext_dc_batch_workspace_bytes.restype = i64
        L.isoext_dc_batch_workspace_bytes.argtypes = [c_int, ctypes.POINTER(McItem)]
        L.isoext_dc_batch_count.restype = c_int
        L.isoext_dc_batch_count.argtypes = [c_int, ctypes.POINTER(McItem), vp, i64, ctypes.POINTER(i64), vp]
        L.isoext_dc_batch_scratch_bytes.restype = i64
        L.isoext_dc_batch_scratch_bytes.argtypes = [c_int, ctypes.POINTER(McItem), ctypes.POINTER(i64)]
        L.isoext_dc_batch_run.restype = c_int
        L.isoext_dc_batch_run.argtypes = [c_int, ctypes.POINTER(McItem), ctypes.POINTER(i64), ctypes.c_float,
                                          ctypes.c_float, vp, i64, vp, i64, vp, i64, vp, i64, ctypes.POINTER(i64),
                                          vp]
        _declared = True
        return L


@dataclass
class GridJob:
    """One extraction of a batch: a stored grid (values), or the field of an
    SDF program (sdf: a csg.SdfProgram, values None, shape given) evaluated
    inside the kernels; sdf_normals: dual contouring with the program's
    analytic normals instead of trilinear ones."""

    values: torch.Tensor | None
    level: float = 0.0
    method: int = 0
    aabb_min: tuple = (-1.0, -1.0, -1.0)
    aabb_max: tuple = (1.0, 1.0, 1.0)
    sdf: object = None
    shape: tuple | None = None
    sdf_normals: bool = False

    @property
    def grid_shape(self) -> tuple:
        return tuple(int(s) for s in (self.values.shape if self.sdf is None else self.shape))

    @property
    def device(self):
        return self.values.device if self.sdf is None else self.sdf.device


BATCH_SPECIAL_CAP = 4096


def _items(jobs, who):
    dev = jobs[0].device
    items = (McItem * len(jobs))()
    for it, j in zip(items, jobs):
        t = j.values
        if j.sdf is not None:
            if j.sdf.device != dev or j.shape is None or len(j.shape) != 3:
                raise TypeError(f"{who}: an SDF job needs a program on the batch's device and a 3-entry shape")
            it.sdf = j.sdf.ptr
            it.sdf_normals = 1 if j.sdf_normals else 0
        else:
            if t.device != dev or t.dtype != torch.float32 or not t.is_contiguous():
                raise TypeError(f"{who}: values must be contiguous float32 tensors on one device")
            it.values = t.data_ptr()
        it.shape[:] = j.grid_shape[:3]
        it.aabb_min[:] = [float(a) for a in j.aabb_min[:3]]
        it.aabb_max[:] = [float(a) for a in j.aabb_max[:3]]
        it.level = float(j.level)
        it.method = int(j.method)
    return dev, items


MAX_DC_BATCH = 256


def dc_batch(jobs: list[GridJob], reg: float = 1e-2, svd_tol: float = 1e-6, ws_kind: str = "dc_batch",
             on_sizes=None):
    """Dual contouring (intersections with trilinear normals, then the QEF
    solve) over a ragged list of dense grids, at most 256 per call.  Returns
    a list of (v, f) pairs, (None, None) for an empty mesh, as
    ``dual_contouring(grid, level, reg=reg, svd_tol=svd_tol)`` per grid.
    on_sizes(out_bytes), if given, receives after phase 1 the output bytes
    each grid's mesh buffers take (12 per active cell, 24 per intersection)."""
    if not jobs:
        return []
    if len(jobs) > MAX_DC_BATCH:
        return (dc_batch(jobs[:MAX_DC_BATCH], reg, svd_tol, ws_kind, on_sizes) +
                dc_batch(jobs[MAX_DC_BATCH:], reg, svd_tol, ws_kind, on_sizes))
    L = _decl()
    dev, items = _items(jobs, "dc_batch")
    for it in items:
        it.method = 0   # not used by dual contouring
    n = len(jobs)
    counts = (ctypes.c_int64 * (2 * n))()
    out_counts = (ctypes.c_int64 * (4 * n + 1))()
    stream = _lib.stream_ptr(dev)
    with torch.cuda.device(dev):
        ws_bytes = L.isoext_dc_batch_workspace_bytes(n, items)
        if ws_bytes < 0:
            raise ValueError(_lib.last_error())
        ws = workspace.get(ws_kind, ws_bytes, dev)
        _lib.check(L.isoext_dc_batch_count(n, items, ws.data_ptr(), ws.numel(), counts, stream), "dc_batch count")
        C = sum(int(counts[2 * i]) for i in range(n))
        P = sum(int(counts[2 * i + 1]) for i in range(n))
        if on_sizes is not None:
            on_sizes([12 * int(counts[2 * i]) + 24 * int(counts[2 * i + 1]) for i in range(n)])
        if C == 0:
            return [(None, None)] * n
        sc = workspace.get(ws_kind + "_scratch", L.isoext_dc_batch_scratch_bytes(n, items, counts), dev)
        out_v = torch.empty((C, 3), dtype=torch.float32, device=dev)
        out_f = torch.empty((max(2 * P, 1), 3), dtype=torch.int32, device=dev)
        rc = L.isoext_dc_batch_run(n, items, counts, float(reg), float(svd_tol), ws.data_ptr(), ws.numel(),
                                   sc.data_ptr(), sc.numel(), out_v.data_ptr(), out_v.shape[0], out_f.data_ptr(),
                                   out_f.shape[0], out_counts, stream)
    _lib.check(rc, "dc_batch")
    res = []
    for i in range(n):
        nv, nf, v0, f0 = (int(out_counts[4 * i + k]) for k in range(4))
        if nf == 0:
            res.append((None, None))
            continue
        v, f = out_v[v0:v0 + nv], out_f[f0:f0 + nf]
        if n == 1:   # one grid: do not pin buffers sized for the worst case behind a smaller mesh
            if out_v.shape[0] > 2 * nv + (1 << 16):
                v = v.clone()
            if out_f.shape[0] > 2 * nf + (1 << 16):
                f = f.clone()
        res.append((v, f))
    return res


# Emit tile configuration of batches (16 x 16 cell rows x 2 words): all
# grids' tiles share one launch, so the single-grid rule (enough tiles to
# fill the GPU) does not apply; this configuration measured fastest over the
# serving mix of 32^3 to 512^3 grids (12% below each grid's own choice).
BATCH_CFG = 2


def mc_batch(jobs: list[GridJob], cfg: int | None = BATCH_CFG, ws_kind: str = "mc_batch", on_sizes=None):
    """Marching cubes over a ragged list of dense grids.  Returns a list of
    (v, f) pairs (zero-row tensors for empty meshes).  cfg: one emit tile
    configuration for every grid (default BATCH_CFG), or None for each
    grid's own (isoext_mc_auto_config).  on_sizes(out_bytes), if given,
    receives after phase 1 each grid's output bytes (12 per provisional
    vertex and face)."""
    if not jobs:
        return []
    L = _decl()
    n = len(jobs)
    dev, items = _items(jobs, "mc_batch")
    if cfg is None:
        cfg = -1   # each grid uses its own tile configuration
    special = BATCH_SPECIAL_CAP
    counts = (ctypes.c_int64 * (2 * n))()
    stream = _lib.stream_ptr(dev)
    with torch.cuda.device(dev):
        ws_bytes = L.isoext_mc_batch_workspace_bytes(n, items, cfg, special)
        if ws_bytes < 0:
            raise ValueError(_lib.last_error())
        ws = workspace.get(ws_kind, ws_bytes, dev)
        _lib.check(L.isoext_mc_batch_count(n, items, cfg, ws.data_ptr(), ws.numel(), special, counts, stream),
                   "mc_batch count")
        # one vertex and one face buffer for the batch; each grid gets a slice
        nvs, nfs = counts[0::2], counts[1::2]
        if on_sizes is not None:
            on_sizes([12 * a + 12 * b for a, b in zip(nvs, nfs)])
        all_v = torch.empty((max(sum(nvs), 1), 3), dtype=torch.float32, device=dev)
        all_f = torch.empty((max(sum(nfs), 1), 3), dtype=torch.int32, device=dev)
        pv, pf = all_v.data_ptr(), all_f.data_ptr()
        for it, a, b in zip(items, nvs, nfs):
            it.out_v, it.cap_v, it.out_f, it.cap_f = pv, a, pf, b
            pv += 12 * a
            pf += 12 * b
        rc = L.isoext_mc_batch_emit(n, items, cfg, ws.data_ptr(), ws.numel(), special, counts, stream)
    _lib.check(rc, "mc_batch emit")
    res = []
    vs, fs = _pieces(all_v, counts[0::2], nvs), _pieces(all_f, counts[1::2], nfs)
    for j, v, f, nv in zip(jobs, vs, fs, counts[0::2]):
        if nv < 0:   # special lists overflowed the batch capacity: run this grid alone
            from .mc import mc_dense_raw
            v, f, _ = mc_dense_raw(j.values, j.grid_shape, j.aabb_min, j.aabb_max, j.level, j.method,
                                   cfg if cfg >= 0 else None, program=j.sdf)
        res.append((v, f))
    return res


def _pieces(buf, used, room):
    """The first used[i] rows of each room[i] rows of buf (none if used[i] is
    negative), from one call.  The unsafe split: autograd lets its pieces be
    changed in place, and they never share a row."""
    sizes = []
    for u, r in zip(used, room):
        u = max(u, 0)
        sizes += (u, r - u)
    return buf.unsafe_split_with_sizes([*sizes, buf.shape[0] - sum(room)])[:-1:2]
