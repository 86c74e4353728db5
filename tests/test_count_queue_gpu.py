"""Count pass that queues the crossed chunks: the oracle's mesh on grids of
at least 512 and 2048 count blocks, with the surface on the last points of
words, rows, slabs and of the grid, and with every chunk empty, full or
crossed."""

import numpy as np
import pytest

from test_mc_dense_gpu import assert_same_mesh

pytestmark = pytest.mark.gpu

# (rows of 1024 a block) 512 and 2048 blocks and a remainder; Z with and without a part word, one word and two
SHAPES = [(750, 701, 2), (1025, 513, 64), (725, 724, 65), (1450, 1449, 3)]


def field(kind, shape):
    v = np.full(shape, 1.0, np.float32)
    if kind == "full":
        v[:] = -1.0
    elif kind == "last":      # the last point of the grid, of a row, of a word; the first of the next word
        v[-1, -1, -1] = v[7, 9, -1] = v[300, -1, min(63, shape[2] - 1)] = -1.0
        if shape[2] > 64:
            v[20, 21, 64] = -0.5
            v[40:42, 30:33, :64] = -0.25   # words set, the next point clear
    elif kind == "lone":      # an outside point in a full grid, next to row and slab ends
        v[:] = -1.0
        v[-1, 4, 0] = v[5, -1, 0] = v[0, 0, -1] = 1.0
    return v


@pytest.mark.parametrize("shape", SHAPES)
@pytest.mark.parametrize("kind", ["empty", "full", "last", "lone"])
def test_sparse_masks(gpu, kind, shape):
    assert_same_mesh(field(kind, shape))


@pytest.mark.parametrize("shape", [(760, 700, 2), (1460, 1450, 2)])
def test_every_chunk_crossed(gpu, shape):
    v = np.random.default_rng(7).standard_normal(shape).astype(np.float32)
    assert_same_mesh(v)
