"""Parser's lists by pyseqm_pair_lists against its general way (taken on the CPU, and for other types, layouts, cutoffs)
for ragged batches, single atoms, empty rows and the calls that must keep the general way.  Whole numbers are equal;
distances and unit vectors are three products and a root: 4 eps."""
import types

import numpy as np
import pytest
import torch

from pyseqm_amd.basics import Parser
from pyseqm_amd.seqm_functions.constants import Constants

pytestmark = pytest.mark.gpu
DEV = "cuda"
SHAPES = {"one": [[6, 1, 1, 1, 1]], "ragged": [[8, 1, 1, 0, 0], [6, 6, 6, 1, 1], [1, 1, 0, 0, 0], [8, 0, 0, 0, 0]],
          "atoms": [[8], [6]], "blank row": [[0, 0, 0], [1, 1, 0]],
          "wide": [[6] * 66 + [1] * 4, [6] * 2 + [0] * 68, [8] * 65 + [0] * 5]}


def _molecule(sp, xyz, const, dev):
    return types.SimpleNamespace(species=sp.to(dev), coordinates=xyz.to(dev), const=const, tot_charge=0)


def _run(sp, xyz, dev, cutoff=None):
    p = {"elements": [0, 1, 6, 8]}
    if cutoff is not None:
        p["pair_outer_cutoff"] = cutoff
    mol = _molecule(sp, xyz, Constants().to(dev), dev)
    parser = Parser(p)
    return parser(mol, "AM1", return_mask_l=True), (parser._lists_on_device(mol) if dev == DEV else None)


def _compare(got, want):
    assert len(got) == len(want)
    for a, b in zip(got, want):
        if not torch.is_tensor(b):
            assert a == b
            continue
        a = a.cpu()
        assert a.shape == b.shape and a.dtype == b.dtype
        if b.dtype.is_floating_point:
            assert torch.allclose(a, b, rtol=1e-15, atol=1e-15, equal_nan=True)
        else:
            assert torch.equal(a, b)


@pytest.mark.parametrize("name", sorted(SHAPES))
@pytest.mark.parametrize("form", ["plain", "int32", "float32", "strided", "cutoff", "nan"])
def test_lists_match_the_general_way(name, form):
    sp = torch.tensor(SHAPES[name], dtype=torch.int64)
    xyz = torch.as_tensor(np.random.default_rng(2).normal(size=tuple(sp.shape) + (3,)) * 3.0)
    cutoff, fast = None, True
    if form == "int32":
        sp, fast = sp.int(), False
    elif form == "float32":
        xyz, fast = xyz.float(), False
    elif form == "strided":
        xyz = xyz.transpose(0, 1).contiguous().transpose(0, 1)
        fast = xyz.is_contiguous()
    elif form == "cutoff":
        cutoff = 4.0
    elif form == "nan":
        xyz[-1, 0, 0] = float("nan")
    got, lists = _run(sp, xyz, DEV, cutoff)
    want, _ = _run(sp, xyz, "cpu", cutoff)
    if form in ("cutoff", "nan"):  # every pair kept, or the general way
        n = int(((sp > 0).sum(1) * ((sp > 0).sum(1) - 1) // 2).sum())
        fast = len(want[-1]) == n
    assert (lists is not None) == fast
    tol = want if form != "float32" else [w for w in want]
    if form == "float32":
        for a, b in zip(got, tol):
            if torch.is_tensor(b) and b.dtype.is_floating_point:
                assert torch.allclose(a.cpu(), b, rtol=1e-6, atol=1e-6)
            elif torch.is_tensor(b):
                assert torch.equal(a.cpu(), b)
    else:
        _compare(got, want)
