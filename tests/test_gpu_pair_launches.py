"""Integrals and forces in one launch over the kinds of pair tiles and in a launch per kind (from 8193 tiles on) give
the same bits for the same molecules."""
import numpy as np
import pytest
import torch

from pyseqm_amd.engine import SCFEngine

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("nmol", [2730, 2731])  # three tiles each: 8190 and 8193
@pytest.mark.parametrize("heavy", [2, 4])
def test_both_launches_agree(nmol, heavy):
    sp = np.array([[6] * heavy + [1] * (8 - heavy)], dtype=np.int64).repeat(nmol, 0)
    rng = np.random.default_rng(heavy)
    base = np.stack(np.meshgrid([0.0, 1.3], [0.0, 1.4], [0.0, 1.5], indexing="ij"), -1).reshape(8, 3)
    xyz = base[None] + rng.uniform(-0.1, 0.1, (nmol, 8, 3))
    out = []
    for n in (nmol, 7):
        eng = SCFEngine(sp[:n], torch.as_tensor(xyz[:n], device=DEV), "PM3", DEV)
        assert (sum(eng.b.ntile) > 8192) == (n == 2731)
        size = int(eng.b.norb[0]) ** 2
        p = np.random.default_rng(1).normal(size=(int(eng.b.norb[0]),) * 2)
        P = torch.as_tensor(np.tile((p + p.T).reshape(-1), n), device=DEV)
        f = eng.forces(P)
        out.append((eng.H[:7 * size], eng.w_reference()[:7 * 28], f[:7 * 8], eng.enuc[:7]))
    for a, c in zip(*out):
        assert torch.equal(a, c)
