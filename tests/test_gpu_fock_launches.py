"""Fock builds of batches that take the pair tiles in one launch, H-H tiles apart, or a launch per kind: copies of one
molecule, so that every molecule's Fock matrix and energy equal those of a small batch bit for bit."""
import numpy as np
import pytest
import torch

from pyseqm_amd.engine import SCFEngine
from pyseqm_amd.layout import PackedBatch

pytestmark = pytest.mark.gpu


def _build(shape, copies, x, P1):
    nh, nH = shape
    b = PackedBatch.from_counts([nh] * copies, [nH] * copies, [(4 * nh + nH) // 2] * copies, nh + nH, "cuda")
    eng = SCFEngine(None, None, "AM1", "cuda", batch=b)
    eng.set_coordinates(x.repeat(copies, 1))
    P = P1.repeat(copies)
    F = torch.full_like(P, float("nan"))
    e = eng.fock(P, F, eelec=torch.full((copies,), float("nan"), dtype=torch.float64, device="cuda"))
    return list(b.ntile), F.view(copies, -1), e


# (heavy atoms, hydrogens), copies: H-H tiles 16380 and 16400 around the limit, no heavy-heavy tiles, hydrogens alone
@pytest.mark.parametrize("shape,copies", [((2, 32), 1638), ((2, 32), 1640), ((9, 26), 1700), ((1, 30), 1700),
                                          ((1, 30), 900), ((0, 26), 40), ((0, 26), 1700)])
def test_launches_agree(shape, copies):
    nh, nH = shape
    n = 4 * nh + nH
    rng = np.random.default_rng(n)
    x = torch.as_tensor(rng.normal(size=(nh + nH, 3)) * 4.0, device="cuda")
    P1 = rng.normal(size=(n, n))
    P1 = torch.as_tensor((P1 + P1.T).reshape(-1), device="cuda")
    tiles, F, e = _build(shape, copies, x, P1)
    few, F1, e1 = _build(shape, 2, x, P1)
    assert [t * copies for t in few] == [2 * t for t in tiles]
    assert bool(torch.isfinite(F1).all()) and bool(torch.isfinite(e1).all())
    assert torch.equal(F, F1[:1].expand_as(F)) and torch.equal(e, e1[:1].expand_as(e))
