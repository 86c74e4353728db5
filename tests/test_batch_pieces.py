"""Meshes of a batch are cut from one buffer; each can be changed in place
with a tensor that autograd tracks, as a single grid's mesh can."""

import torch

from isoext_amd.batch import _pieces


def test_pieces_and_in_place_gradients():
    buf = torch.arange(36, dtype=torch.float32).reshape(12, 3)
    want = buf.clone()
    used, room = [3, -1, 0, 2], [4, 2, 0, 5]   # an unused row, a negative count, an empty piece, a rest
    got = _pieces(buf, used, room)
    assert [p.shape[0] for p in got] == [3, 0, 0, 2]
    assert torch.equal(got[0], want[0:3]) and torch.equal(got[3], want[6:8])
    assert got[3].data_ptr() == buf[6:].data_ptr()
    shift = torch.ones(3, 3, requires_grad=True)
    got[0].add_(2 * shift)
    got[0].sum().backward()
    assert torch.equal(shift.grad, torch.full((3, 3), 2.0)) and torch.equal(got[0].detach(), want[0:3] + 2)
    assert not got[3].requires_grad and torch.equal(got[3], want[6:8])
