"""Rows are moved through pointers only where nothing else has to follow them: a tangent, a batch dimension, a trace."""

import torch
from torch._subclasses.fake_tensor import FakeTensorMode

from nvalchemi_amd import _lib
from nvalchemi_amd.data import batch as batch_module


def test_transforms_take_the_general_way():
    seen = []
    assert _lib.plainly_eager()
    torch.func.vmap(lambda x: seen.append(_lib.plainly_eager()) or x)(torch.ones(2, 3))
    torch.func.jvp(lambda x: seen.append(_lib.plainly_eager()) or x, (torch.ones(2),), (torch.ones(2),))
    with torch.autograd.forward_ad.dual_level():
        seen.append(_lib.plainly_eager())
    with FakeTensorMode():
        seen.append(_lib.plainly_eager())
    assert seen == [False] * 4 and _lib.plainly_eager()


def test_a_selection_keeps_its_tangent():
    with torch.autograd.forward_ad.dual_level():
        dual = torch.autograd.forward_ad.make_dual(torch.ones(3, 2), torch.full((3, 2), 2.0))
        (out,) = batch_module._copies([dual[1:]])
        assert (torch.autograd.forward_ad.unpack_dual(out).tangent == 2.0).all()
