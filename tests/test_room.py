"""Room that intersections and dual contouring of a dense grid start with:
never more than the grid can hold, however flat it is, and no more than a
few million cells on a guess."""

import pytest

from isoext_amd import dc


def cells(shape):
    return (shape[0] - 1) * (shape[1] - 1) * (shape[2] - 1)


# flat grids have fewer cells than twice their cross-section; the last would pass 2^30 cells
FLAT = [(2, 20000, 20000), (23200, 2, 23200), (30000, 30000, 2), (2, 2, 2), (2, 3, 64), (5, 5, 5), (40000, 40000, 2)]


@pytest.mark.parametrize("shape", FLAT + [(1024, 1024, 1024), (1, 7, 9)])
def test_first_room(monkeypatch, shape):
    monkeypatch.setattr(dc, "_its_hint", {})
    monkeypatch.setattr(dc, "_dc_hint", {})
    most = max(cells(shape), 1)
    nc, npt = dc._its_caps(shape)
    assert 1 <= nc <= min(most, 1 << 22) and nc <= npt <= 12 * most
    nc, cap_v, cap_f = dc._dc_caps(shape)
    assert 1 <= nc <= min(most, 1 << 22) and cap_v <= nc and cap_f <= 2 * nc


@pytest.mark.parametrize("shape", FLAT)
def test_room_after_a_full_grid(monkeypatch, shape):
    most = cells(shape)
    monkeypatch.setattr(dc, "_its_hint", {shape: (most, 12 * most)})
    monkeypatch.setattr(dc, "_dc_hint", {shape: (most, most, 6 * most)})
    assert dc._its_caps(shape) == (most, 12 * most)
    lim = min(most, 0x3fffffff)   # isoext_dc_grid's own limit
    assert dc._dc_caps(shape) == (lim, lim, 6 * lim)


def test_grid_workspace_per_cell():
    """Lookup tables stand in for the active-cell hash: a cell takes its vertex, flags, ids and place in the scan
    (about 40 B) and two to four position slots of 4 B, not another 24 to 48 B of hash."""
    import ctypes

    from isoext_amd import _lib
    g = dc.IsoGrid()
    g.values = 64   # any address: sizes only
    for a in range(3):
        g.shape[a], g.aabb_min[a], g.aabb_max[a] = 1024, -1.0, 1.0
    size = _lib.lib().isoext_dc_grid_workspace_bytes
    n = 1 << 20
    assert (size(ctypes.byref(g), 2 * n) - size(ctypes.byref(g), n)) / n < 60


def test_sizes_that_vary(monkeypatch):
    """Counted first only while small sets are among the recent ones: a steady size is guessed again soon, also after
    empty sets."""
    for name in ("_its_hint", "_its_low"):
        monkeypatch.setattr(dc, name, {})
    shape, vary = (200, 200, 200), []
    for n in [0, 0] + [400_000] * 9 + [2_000] + [400_000] * 9:
        vary.append(dc._its_vary(shape))
        dc._remember(dc._its_hint, shape, (n // 4, n), dc._its_low)
    assert not any(vary[:3]) and all(vary[3:5]) and not any(vary[9:12]) and all(vary[12:14]) and not any(vary[18:])
    for _ in range(200):   # a lone large set is forgotten
        dc._remember(dc._its_hint, shape, (500, 2_000), dc._its_low)
    assert not dc._its_vary(shape) and dc._its_caps(shape)[1] < 20_000
