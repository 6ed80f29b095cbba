"""Integrals and forces on both sides of the rules that choose one launch over the kinds of pair tiles or a launch per
kind, by the light tiles beside heavy-heavy ones and without those: the same bits for the same molecules."""
import numpy as np
import pytest
import torch

from pyseqm_amd.engine import SCFEngine

pytestmark = pytest.mark.gpu
DEV = "cuda"


# (heavy atoms, hydrogens), molecules: light tiles 3072 / 3074 without heavy-heavy ones, 6116 / 6160 with them, H-H
# alone
@pytest.mark.parametrize("heavy,hydro,nmol", [(1, 7, 1536), (1, 7, 1537), (2, 62, 139), (2, 62, 140), (0, 8, 9),
                                              (0, 8, 3100)])
def test_launches_agree(heavy, hydro, nmol):
    n = heavy + hydro
    sp = np.array([[6] * heavy + [1] * hydro], dtype=np.int64).repeat(nmol, 0)
    rng = np.random.default_rng(n)
    side = int(np.ceil(n ** (1 / 3)))
    base = np.stack(np.meshgrid(*[np.arange(side) * 1.4] * 3, indexing="ij"), -1).reshape(-1, 3)[:n]
    xyz = base[None] + rng.uniform(-0.1, 0.1, (nmol, n, 3))
    charges = np.full(nmol, (4 * heavy + hydro) % 2)
    out = []
    for m in (nmol, 7):
        eng = SCFEngine(sp[:m], torch.as_tensor(xyz[:m], device=DEV), "PM3", DEV, charges=charges[:m])
        norb = int(eng.b.norb[0])
        p = np.random.default_rng(1).normal(size=(norb, norb))
        P = torch.as_tensor(np.tile((p + p.T).reshape(-1), m), device=DEV)
        f = eng.forces(P)
        out.append((eng.H[:7 * norb * norb], eng.w_reference()[:7 * (n * (n - 1) // 2)], f[:7 * n], eng.enuc[:7]))
    for a, c in zip(*out):
        assert bool(torch.isfinite(a).all()) and torch.equal(a, c)
