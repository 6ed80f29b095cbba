"""Forward-mode derivatives through the padded views: a tensor that carries a tangent takes the index arrays, as one
that requires grad does, and its tangent is viewed like its value (a view is linear)."""
import types

import numpy as np
import pytest
import torch
import torch.autograd.forward_ad as fwad

from pyseqm_amd.layout import PackedBatch

SP = np.array([[6, 6, 1, 1, 1, 0], [8, 1, 1, 0, 0, 0]])


def test_a_tangent_is_not_plain():
    # a device batch as far as this rule looks, on the CPU
    b = types.SimpleNamespace(device=torch.device("cuda"), d={"mol_norb": torch.zeros(1)})
    x = torch.zeros(4, dtype=torch.float64)
    assert PackedBatch._plain(b, x)
    with fwad.dual_level():
        assert PackedBatch._plain(b, x)
        assert not PackedBatch._plain(b, fwad.make_dual(x, torch.ones_like(x)))


@pytest.mark.parametrize("device", ["cpu", pytest.param("cuda", marks=pytest.mark.gpu)])
def test_tangents_pass(device):
    b = PackedBatch(SP, "AM1", torch.device(device), np.array([1, 0]))
    g = torch.Generator().manual_seed(4)
    w = 4 * b.molsize
    for view, shape in ((b.to_padded, (b.total,)), (b.from_padded, (b.nmol, w, w))):
        x, t = (torch.randn(shape, dtype=torch.float64, generator=g).to(device) for _ in range(2))
        with fwad.dual_level():
            out = fwad.unpack_dual(view(fwad.make_dual(x, t)))
            assert torch.equal(out.primal, view(x)) and torch.equal(out.tangent, view(t))
        val, tan = torch.func.jvp(view, (x,), (t,))
        assert torch.equal(val, view(x)) and torch.equal(tan, view(t))
