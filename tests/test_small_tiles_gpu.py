"""Emit tiles of 4 x 4 x 64 cells, the choice for grids of few tiles: the
same arrays as from 8 x 8 x 64 tiles and the oracle's mesh, at tile, word
and wave edges and on both sides of the rule's line."""

import numpy as np
import pytest

from conftest import multi_sphere_field
from test_mc_dense_gpu import assert_same_mesh, run_gpu

SMALL, WIDE = 7, 5


def test_rule():
    from isoext_amd import _lib
    auto = _lib.lib().isoext_mc_auto_config
    assert auto(_lib.i64x3((18, 5, 2))) == auto(_lib.i64x3((192, 192, 192))) == SMALL
    # 27 * 26 * 3 = 2106 tiles of 8 x 8 x 64, 26 * 26 * 3 = 2028
    assert auto(_lib.i64x3((217, 209, 193))) == WIDE
    assert auto(_lib.i64x3((209, 209, 193))) == SMALL


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
