"""Dual vertices do not depend on the length of the caller's normals: normals
times 2^k with the regularisation times 4^k are the same minimisation times
4^k.  Both solutions are within 1e-4 cell sizes of its FP64 minimum (the
bound of the oracle comparison), so they differ by at most twice that."""

import numpy as np
import pytest

from conftest import multi_sphere_field

pytestmark = pytest.mark.gpu


# 2^32 and up: the squares of the QEF matrix's entries overflow in FP32, from 2^48 also those of its trace; 2^60: close to
# where the matrix does.  2^-40 and below: they vanish
@pytest.mark.parametrize("k", [-50, -40, 10, 33, 48, 50, 60])
def test_scaled_normals(gpu, k):
    import torch

    import isoext_amd as iso
    from isoext_amd import dc
    shape = (24, 21, 33)
    g = iso.UniformGrid.wrap(torch.from_numpy(multi_sphere_field(shape, 6, seed=5)).cuda())
    its = iso.get_intersection(g, 0.03, True)
    one = dc.dc_raw(g, its, its.normals, 1e-2, 1e-6, want_dual=True)[3]
    dual = dc.dc_raw(g, its, its.normals * 2.0 ** k, 1e-2 * 4.0 ** k, 1e-6, want_dual=True)[3]
    h = 2.0 / (np.array(shape) - 1).min()
    assert (dual - one).abs().max().item() <= 2e-4 * h
