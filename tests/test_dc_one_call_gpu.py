"""Dual contouring and intersections of a dense grid launched before the
active cells are counted: equal, element for element, to the counted path
whatever room the buffers start with, at wave, workgroup and scan edges."""

import ctypes

import numpy as np
import pytest

from conftest import multi_sphere_field

pytestmark = pytest.mark.gpu


def counted(grid, level, normals):
    """get_intersection by the two-call ABI."""
    import torch

    from isoext_amd import _lib, dc
    L, g, dev = _lib.lib(), dc.grid_struct(grid), grid.values.device
    scratch = torch.zeros(L.isoext_its_scratch_bytes(ctypes.byref(g)), dtype=torch.uint8, device=dev)
    counts, st = (ctypes.c_int64 * 2)(), _lib.stream_ptr(dev)
    assert L.isoext_its_count(ctypes.byref(g), level, scratch.data_ptr(), scratch.numel(), counts, st) == 0
    nc, npt = int(counts[0]), int(counts[1])
    b = dc._its_buffers(nc, npt, normals, dev)
    nt = max(int(L.isoext_its_table_entries(g.shape)), 1)
    tab = (torch.empty(nt, dtype=torch.int64, device=dev), torch.empty(nt, dtype=torch.int32, device=dev))
    assert L.isoext_its_emit(ctypes.byref(g), level, scratch.data_ptr(), nc, npt,
                             *(t.data_ptr() if t is not None else None for t in b), tab[0].data_ptr(),
                             tab[1].data_ptr(), st) == 0
    torch.cuda.synchronize()
    return dc.Intersection(grid, level, *b, tab if nc else None)


def field(kind, shape):
    if kind == "spheres":
        return multi_sphere_field(shape, 6, seed=5)
    if kind == "none":
        return np.full(shape, 1.0, np.float32)
    if kind == "one":   # one cell
        v = np.full(shape, 1.0, np.float32)
        v[0, 0, 0] = -1.0
        return v
    v = np.random.default_rng(sum(shape)).standard_normal(shape).astype(np.float32)
    return np.round(v) if kind == "ties" else v   # ties: vertices on their cells' boxes, welded


# noise: most cells active, up to 12 entries a cell (more than a wave's LDS holds at once); 70^3: more blocks than
# are added up without a scan; the rest: remainders of waves, workgroups and words, and no cell at all
CASES = [("noise", (70, 71, 70)), ("noise", (5, 5, 66)), ("ties", (33, 17, 65)), ("spheres", (48, 40, 72)),
         ("spheres", (9, 80, 129)), ("one", (2, 2, 2)), ("one", (4, 4, 200)), ("none", (16, 9, 5)), ("noise", (1, 7, 9)),
         ("noise", (2, 3, 64))]


@pytest.mark.parametrize("kind,shape", CASES)
@pytest.mark.parametrize("room", ["first", "short", "ample"])
def test_equals_counted(gpu, monkeypatch, kind, shape, room):
    import torch

    import isoext_amd as iso
    from isoext_amd import dc
    g = iso.UniformGrid.wrap(torch.from_numpy(np.ascontiguousarray(field(kind, shape))).cuda())
    level = 0.0 if kind != "spheres" else 0.03
    for hint in (dc._its_hint, dc._dc_hint):
        hint.pop(shape, None)
    if room != "first":
        n = 4 if room == "short" else 1 << 20
        monkeypatch.setattr(dc, "_its_caps", lambda _: (n, n))
        monkeypatch.setattr(dc, "_dc_caps", lambda _: (n, n, n))
    its = iso.get_intersection(g, level, True)
    ref = counted(g, level, True)
    for k in ("cell_indices", "cell_dense", "cell_offsets", "points", "normals", "edge_local", "is_out", "entry_cell"):
        assert torch.equal(getattr(its, k), getattr(ref, k)), k
    v, f = iso.dual_contouring(g, level)
    if len(ref) == 0:
        assert v is None and f is None
        return
    vr, fr, _ = dc.dc_raw(g, ref, ref.normals, 1e-2, 1e-6)
    if fr.shape[0] == 0:
        assert v is None and f is None
    else:
        assert torch.equal(v, vr) and torch.equal(f, fr)
    vi, fi = iso.dual_contouring(g, level, its)
    assert (vi is None and fr.shape[0] == 0) or (torch.equal(vi, vr) and torch.equal(fi, fr))


def test_refusals_and_empty(gpu):
    import torch

    import isoext_amd as iso
    g = iso.UniformGrid([4, 0, 4])
    with pytest.raises(ValueError):
        iso.dual_contouring(g)
    s = iso.SparseGrid([8, 8, 8])
    its = iso.get_intersection(s)
    assert len(its) == 0 and its.cell_offsets.tolist() == [0]
    assert iso.dual_contouring(s) == (None, None)
    torch.cuda.synchronize()


def test_small_and_large_surfaces_in_turn(gpu, monkeypatch):
    """Each is run once: the room for the large one is kept over small ones between."""
    import torch

    import isoext_amd as iso
    from isoext_amd import dc
    shape = (60, 61, 62)
    large = iso.UniformGrid.wrap(torch.from_numpy(field("noise", shape)).cuda())
    small = iso.UniformGrid.wrap(torch.from_numpy(field("spheres", shape)).cuda())
    runs = []
    buffers, get = dc._its_buffers, dc.workspace.get
    monkeypatch.setattr(dc, "_its_buffers", lambda *a: (runs.append("its"), buffers(*a))[1])
    monkeypatch.setattr(dc.workspace, "get", lambda kind, *a: (runs.append(kind), get(kind, *a))[1])
    monkeypatch.setattr(dc, "_its_hint", {})
    monkeypatch.setattr(dc, "_dc_hint", {})
    for g in (large, small, small, small, large, small, large):
        a, b = (dc._its_hint.get(shape), dc._dc_hint.get(shape))
        runs.clear()
        its, mesh = iso.get_intersection(g, 0.0, True), iso.dual_contouring(g, 0.0)
        if a is not None and b is not None:   # the first call knows nothing
            assert runs.count("dc_grid") == 1 and runs.count("its") == 2   # scratch and one set of buffers
        ref = counted(g, 0.0, True)
        assert torch.equal(its.points, ref.points) and torch.equal(its.cell_offsets, ref.cell_offsets)
        assert torch.equal(mesh[0], dc.dc_raw(g, ref, ref.normals, 1e-2, 1e-6)[0])


def test_grids_without_a_cell_in_turn(gpu, monkeypatch):
    """After a grid without a cell the next of its shape is counted first."""
    import torch

    import isoext_amd as iso
    from isoext_amd import dc
    shape = (20, 21, 66)
    none, some = (iso.UniformGrid.wrap(torch.from_numpy(field(k, shape)).cuda()) for k in ("none", "spheres"))
    v, f = iso.dual_contouring(some, 0.03)
    runs, caps = [], dc._dc_caps
    monkeypatch.setattr(dc, "_dc_caps", lambda s: (runs.append(s), caps(s))[1])
    monkeypatch.setattr(dc, "_dc_hint", {})
    monkeypatch.setattr(dc, "_dc_none", set())
    for g, run in ((none, 1), (none, 0), (none, 0), (some, 1), (some, 1), (none, 1), (none, 0), (some, 1)):
        runs.clear()
        a, b = iso.dual_contouring(g, 0.03)
        assert len(runs) == run
        assert a is None and b is None if g is none else torch.equal(a, v) and torch.equal(b, f)


def test_begun_and_given_up(gpu, monkeypatch):
    """A set that was begun and given up has written its counts before the thread's next one is begun, on any stream."""
    import torch

    import isoext_amd as iso
    from isoext_amd import dc
    a, b = (iso.UniformGrid.wrap(torch.from_numpy(field("spheres", s)).cuda()) for s in ((30, 31, 32), (20, 21, 22)))
    ref = counted(b, 0.0, True)
    iso.get_intersection(a, 0.0, True)
    first, second = torch.cuda.Stream(), torch.cuda.Stream()
    for s in (first, second):   # workspaces, tables
        with torch.cuda.stream(s):
            iso.get_intersection(b, 0.0, True)
    torch.cuda.synchronize()

    def no_memory(*args):
        raise MemoryError

    with monkeypatch.context() as m, torch.cuda.stream(first):
        torch.cuda._sleep(5_000_000)
        m.setattr(dc, "_its_buffers", no_memory)
        with pytest.raises(MemoryError):
            iso.get_intersection(a, 0.0, True)
    with torch.cuda.stream(second):
        its = iso.get_intersection(b, 0.0, True)
    assert first.query()
    torch.cuda.synchronize()
    assert torch.equal(its.points, ref.points) and torch.equal(its.cell_offsets, ref.cell_offsets)
