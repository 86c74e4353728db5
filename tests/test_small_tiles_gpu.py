"""Emit tiles of 4 x 4 x 64 cells, the choice for grids of few tiles: the
same arrays as from 8 x 8 x 64 tiles and the oracle's mesh, at tile, word
and wave edges and on both sides of the rule's line."""

import numpy as np
import pytest

from conftest import multi_sphere_field
from test_mc_dense_gpu import assert_same_mesh, run_gpu

SMALL, WIDE = 7, 5


# at most 512 tiles of 8 x 8 x 64 cells, of more than 256 cells each: (18, 5, 2) has tiles of 8 x 4 x 1,
# 128^3 512 tiles, (129, 137, 129) 544, (120, 120, 5) tiles of 256 cells and (120, 120, 6) of 320; flat grids and
# larger ones keep the wide tiles
@pytest.mark.parametrize("shape,small", [
    ((64, 64, 64), True), ((97, 131, 75), True), ((128, 128, 128), True), ((129, 129, 129), True),
    ((129, 137, 129), False), ((120, 120, 6), True), ((120, 120, 5), False), ((160, 160, 33), True),
    ((200, 200, 33), False), ((362, 362, 2), False), ((300, 400, 2), False), ((2, 8192, 16), False),
    ((2, 1024, 128), True), ((2, 2049, 129), True), ((2, 2058, 129), False), ((192, 192, 192), False),
    ((256, 256, 65), False), ((18, 5, 2), False), ((2, 2, 2), False), ((10, 10, 10), True)])
def test_rule(shape, small):
    """What marching cubes takes (table or rule) and what intersections take (the rule)."""
    from isoext_amd import _lib, autotune
    assert (_lib.lib().isoext_mc_auto_config(_lib.i64x3(shape)) == SMALL) == small
    assert (autotune.mc_config(shape) == SMALL) == small


# noise fills tiles (1024 cells, four rounds of a workgroup), ties weld
@pytest.mark.gpu
@pytest.mark.parametrize("kind", ["noise", "ties", "spheres"])
@pytest.mark.parametrize("shape", [(2, 2, 2), (5, 5, 65), (6, 4, 66), (4, 9, 64), (33, 18, 129), (64, 64, 64)])
def test_equals_wide_and_oracle(gpu, kind, shape):
    v = multi_sphere_field(shape, 4, seed=3) if kind == "spheres" else \
        np.random.default_rng(sum(shape)).standard_normal(shape).astype(np.float32)
    if kind == "ties":
        v = np.round(v)
    for method in ("nagae", "lorensen"):
        assert_same_mesh(v, 0.0, method, cfg=SMALL)
        a, b = run_gpu(v, 0.0, method, cfg=SMALL), run_gpu(v, 0.0, method, cfg=WIDE)
        assert all(np.array_equal(np.asarray(x), np.asarray(y)) for x, y in zip(a[:2], b[:2]))
