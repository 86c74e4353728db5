"""Sparse marching cubes where its runs and lists can go wrong: runs of
neighbours longer than the LDS holds, workgroup and block remainders, values
that disagree between cells, vertices at grid points, and the two ways
through the C ABI."""

import ctypes

import numpy as np
import pytest

import oracle

pytestmark = pytest.mark.gpu


def corner_values(field, ids):
    """(N, 8) corner values of the cells `ids` of a grid of point values."""
    X, Y, Z = field.shape
    z, r = ids % (Z - 1), ids // (Z - 1)
    y, x = r % (Y - 1), r // (Y - 1)
    return np.stack([field[x + (k >> 2), y + ((k >> 1) & 1), z + (k & 1)] for k in range(8)], 1).astype(np.float32)


def cells_of(shape, keep, rng):
    n = (shape[0] - 1) * (shape[1] - 1) * (shape[2] - 1)
    ids = np.arange(n, dtype=np.int64)
    return ids if keep == 1.0 else ids[rng.random(n) < keep]


def make(shape, ids, vals):
    import torch

    import isoext_amd as iso
    g = iso.SparseGrid(list(shape))
    g.add_cells(torch.from_numpy(ids).cuda())
    g.set_values(torch.from_numpy(vals).cuda())
    return g


# shape, share of cells present, values: "same" (one value a grid point), "own" (each cell its own), "ties" (rounded:
# many corners on the level).  Columns of 700 cells: three of them exceed the runs' LDS space; 3 cells: less than a
# wave; 1100 cells: block and workgroup remainders.
CASES = [((20, 18, 24), 1.0, "same"), ((6, 5, 700), 1.0, "same"), ((6, 5, 700), 1.0, "ties"), ((4, 4, 120), 0.9, "own"),
         ((12, 11, 10), 0.6, "ties"), ((24, 30, 9), 0.3, "own"), ((2, 2, 4), 1.0, "same"), ((9, 40, 2), 1.0, "same"),
         ((1200, 2, 2), 1.0, "ties")]


@pytest.mark.parametrize("shape,keep,kind", CASES)
@pytest.mark.parametrize("method", ["nagae", "lorensen"])
def test_runs_match_oracle(gpu, shape, keep, kind, method):
    import isoext_amd as iso
    rng = np.random.default_rng([*shape, len(kind)])
    ids = cells_of(shape, keep, rng)
    field = rng.standard_normal(shape)
    if kind == "ties":
        field = np.round(field * 1.5)
    vals = rng.standard_normal((len(ids), 8)).astype(np.float32) if kind == "own" else corner_values(field, ids)
    v, f = iso.marching_cubes(make(shape, ids, vals), 0.0, method)
    vo, fo = oracle.mc_sparse(ids, vals, shape, 0.0, method)
    a, b = oracle.canonical(vo, fo), oracle.canonical(v.cpu().numpy(), f.cpu().numpy())
    assert np.array_equal(a[0], b[0]) and np.array_equal(a[1], b[1])


@pytest.mark.parametrize("shape,keep,kind", CASES[:4])
def test_one_step_abi_and_gradients(gpu, shape, keep, kind):
    """isoext_mc_sparse_count / isoext_mc_sparse give the mesh and sources of
    the two-step calls, and isoext_mc_sparse_backward the gradient of
    isoext_mc_backward (one product is rounded in another order: 4 ulps of a
    term, at most 12 terms a row)."""
    import torch

    from isoext_amd import _lib, autograd  # noqa: F401  (autograd declares the backward entry points)
    from isoext_amd.dc import grid_struct
    from isoext_amd.sparse import mc_sparse
    rng = np.random.default_rng([*shape, len(kind)])
    ids = cells_of(shape, keep, rng)
    vals = rng.standard_normal((len(ids), 8)).astype(np.float32)
    if kind != "own":
        vals = corner_values(np.round(rng.standard_normal(shape) * 1.5) if kind == "ties" else
                             rng.standard_normal(shape), ids)
    grid = make(shape, ids, vals)
    v, f, src, jac = mc_sparse(grid, 0.0, 0, want_jac=True)
    assert bool((src[1:] > src[:-1]).all())
    L, g, n = _lib.lib(), grid_struct(grid), len(ids)
    L.isoext_mc_sparse_workspace_bytes.restype = ctypes.c_int64
    L.isoext_mc_sparse_workspace_bytes.argtypes = [ctypes.c_int64] * 2
    scratch = torch.zeros(n // 256 + 16, dtype=torch.int64, device="cuda")
    ninst = ctypes.c_int64(0)
    assert L.isoext_mc_sparse_count(ctypes.byref(g), 0.0, scratch.data_ptr(), ctypes.byref(ninst), None) == 0
    ws = torch.empty(L.isoext_mc_sparse_workspace_bytes(n, ninst.value), dtype=torch.uint8, device="cuda")
    v2, f2 = torch.empty_like(v), torch.empty_like(f)
    src2, counts = torch.empty_like(src), (ctypes.c_int64 * 2)()
    torch.cuda.synchronize()
    assert L.isoext_mc_sparse(ctypes.byref(g), 0.0, 0, ninst.value, ws.data_ptr(), ws.numel(), v2.data_ptr(),
                              v2.shape[0], f2.data_ptr(), f2.shape[0], src2.data_ptr(), counts, None) == 0
    assert tuple(counts) == (v.shape[0], f.shape[0])
    assert torch.equal(v, v2) and torch.equal(f, f2) and torch.equal(src, src2)
    gv = torch.from_numpy(rng.standard_normal(v.shape).astype(np.float32)).cuda()
    gv[::7, 1] = float("inf")   # a gradient that is not finite counts for nothing
    a, b = torch.zeros_like(grid.values), torch.full_like(grid.values, 7.0)
    torch.cuda.synchronize()
    assert L.isoext_mc_backward(ctypes.byref(g), 0.0, gv.data_ptr(), src.data_ptr(), src.numel(), a.data_ptr(),
                                None) == 0
    assert L.isoext_mc_sparse_backward(n, gv.data_ptr(), src.data_ptr(), jac.data_ptr(), src.numel(), b.data_ptr(),
                                       None) == 0
    torch.cuda.synchronize()
    term = torch.zeros_like(a.double()).view(-1)
    e = src % 12
    corner = torch.tensor([[0, 1, 2, 0, 4, 5, 6, 4, 0, 1, 3, 2], [1, 3, 3, 2, 5, 7, 7, 6, 4, 5, 7, 6]], device="cuda")
    axis = torch.tensor([2, 1, 2, 1, 2, 1, 2, 1, 0, 0, 0, 0], device="cuda")
    ga = gv.gather(1, axis[e][:, None])[:, 0].double().nan_to_num(0.0, 0.0, 0.0).abs()
    for k in range(2):
        term.index_add_(0, 8 * (src // 12) + corner[k][e], ga * jac[:, k].double().nan_to_num(0.0, 0.0, 0.0).abs())
    bound = 16 * 2.0 ** -24 * term.view_as(a) + 1e-37
    assert bool(((a.double() - b.double()).abs() <= bound).all())


@pytest.mark.parametrize("shape,kind", [((92, 86, 80), "ties"), ((90, 2, 3400), "ties"), ((3, 420, 500), "lone")])
def test_many_vertices_at_grid_points(gpu, shape, kind):
    """Enough active cells for workgroups of more than 256 of them, with vertices at grid points in most cells, or in a
    few at the ends of columns and slabs: the first cell of every position by the oracle."""
    import isoext_amd as iso
    rng = np.random.default_rng(shape)
    ids = cells_of(shape, 0.98, rng)
    field = np.round(rng.standard_normal(shape) * 1.5)
    if kind == "lone":
        field = np.where(field == 0, 0.37, field)
        field[0, 0, 0] = field[1, -1, -1] = field[2, 0, -1] = field[1, 7, 0] = field[-1, -1, 5] = 0.0
    vals = corner_values(field, ids)
    v, f = iso.marching_cubes(make(shape, ids, vals), 0.0)
    a, b = oracle.canonical(*oracle.mc_sparse(ids, vals, shape, 0.0, "nagae")), oracle.canonical(v.cpu().numpy(),
                                                                                                  f.cpu().numpy())
    assert np.array_equal(a[0], b[0]) and np.array_equal(a[1], b[1])


@pytest.mark.parametrize("n", [16, 44])   # below and above the crossing edges from which buffers are made to size
def test_what_is_kept_for_backward(gpu, monkeypatch, n):
    """Large results are kept at their own size, and are those of a call with room for every crossing edge."""
    import torch

    from isoext_amd import autograd, sparse
    from isoext_amd.sparse import mc_sparse
    monkeypatch.setattr(sparse, "_EXACT_FROM", 1 << 18, raising=False)
    shape, rng = (n, n + 1, n + 2), np.random.default_rng(n)
    ids = cells_of(shape, 1.0, rng)
    grid = make(shape, ids, corner_values(rng.standard_normal(shape), ids))
    values = grid.values.clone().requires_grad_()
    v, f = autograd.marching_cubes(grid, values, 0.0)
    src, jac = v.grad_fn.saved_tensors[1:]
    v2, f2, src2 = mc_sparse(grid, 0.0, 0, want_src=True)
    assert torch.equal(v.detach(), v2) and torch.equal(f, f2) and torch.equal(src, src2)
    kept = sum(t.untyped_storage().nbytes() for t in (src, jac))
    assert kept <= (16 * v.shape[0] if n == 44 else 16 << 18)
    (g,) = torch.autograd.grad(v.sum(), values)
    assert bool(g.isfinite().all()) and g.abs().sum() > 0
