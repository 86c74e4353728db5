"""Count pass that queues the crossed chunks: the oracle's mesh on grids of
at least 512 and 2048 count blocks, with the surface on the last points of
words, rows, slabs and of the grid, and with every chunk empty, full or
crossed; the oracle's counts and intersections where those queue as well."""

import numpy as np
import pytest

import oracle
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


# 2067 and 2050 blocks: from 2048 on intersections queue too (their counts come from the crossing edges, not from the
# dealt triangles)
ITS = [("last", (1460, 1450, 3)), ("lone", (1460, 1450, 3)), ("noise", (1460, 1450, 2)), ("last", (1050, 1000, 66)),
       ("lone", (1050, 1000, 66))]


def its_field(kind, shape):
    if kind == "noise":
        return np.random.default_rng(7).standard_normal(shape).astype(np.float32)
    return field(kind, shape)


@pytest.mark.parametrize("kind,shape", ITS)
def test_intersections(gpu, kind, shape):
    import torch

    import isoext_amd as iso
    v = its_field(kind, shape)
    its = iso.get_intersection(iso.UniformGrid.wrap(torch.from_numpy(v).cuda()), 0.0)
    ref = oracle.intersection(v, 0.0)
    assert np.array_equal(its.cell_indices.cpu().numpy(), ref["cell_indices"])
    assert np.array_equal(its.cell_offsets.cpu().numpy(), ref["cell_offsets"])
    assert np.array_equal(its.get_points().cpu().numpy(), ref["points"])
    assert np.array_equal(its.is_out.cpu().numpy().astype(bool), ref["is_out"])


def test_batch_counts(gpu):
    """Cells and points of each grid of a batch that queues (2067 blocks and more together) are the oracle's."""
    import torch

    from isoext_amd.batch import GridJob, dc_batch
    fields = [its_field("noise", (9, 8, 70)), its_field("last", (1000, 1450, 3)), its_field("lone", (460, 1450, 2)),
              its_field("lone", (400, 300, 66)), its_field("noise", (300, 301, 2))]
    sizes = []
    dc_batch([GridJob(torch.from_numpy(v).cuda()) for v in fields], on_sizes=sizes.append)
    refs = [oracle.intersection(v, 0.0) for v in fields]
    assert sizes[0] == [12 * len(r["cell_indices"]) + 24 * len(r["points"]) for r in refs]
