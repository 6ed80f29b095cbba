"""Closed-form parameter gradients (pyseqm_param_grad) on the overlap formulas and tile shapes that the C, N, O, H
batch of test_gpu_param_grad.py does not meet: second- with third-row pairs, third-row pairs, hydrides of both, and
a molecule over several 8 x 8 tiles.  Against the oracle's 4th-order differences at the same random density; the bar
is that file's, 1e-6 (1 + |d|), 2e-5 (1 + |d|) where equal exponents force a 1e-7 step."""
import numpy as np
import pytest
import torch

from oracle import seqm_ref as R
from pyseqm_amd import workloads as W
from pyseqm_amd.engine import SCFEngine
from pyseqm_amd.seqm_functions.parameters import COLUMNS
from tests.test_gpu_param_grad import _fixed_density_energy

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _check(sp, c, method, seed, names):
    eng = SCFEngine(sp, c, method, DEV)
    b = eng.b
    rng = np.random.default_rng(seed)
    P = torch.zeros_like(eng.H)
    for m in range(b.nmol):
        n, o = int(b.norb[m]), int(b.mol_mat_off[m])
        a = 0.3 * rng.normal(size=(n, n))
        P[o:o + n * n] = torch.as_tensor((a + a.T + np.diag(rng.uniform(0.5, 1.5, n))).reshape(-1), device=DEV)
    G = eng.param_grad(P).cpu().numpy()
    Pp = b.to_padded(P).cpu().numpy()
    ob = R.parse(sp, c, method)
    Zat, mol = np.asarray(b.Z), np.asarray(b.atom_mol)
    for Z in sorted(set(Zat.tolist())):
        sel = Zat == Z
        flat = Z > 1 and ob.prm["zeta_s"][Z] == ob.prm["zeta_p"][Z]
        for name in names:
            base = ob.prm[name][Z]
            short = flat and name in ("zeta_s", "zeta_p")
            h = 1e-7 if short else 1e-4 * max(abs(base), 0.1)
            bar = 2e-5 if short else 1e-6
            ev = []
            for s in (-2, -1, 1, 2):
                ob.prm[name][Z] = base + s * h
                ev.append(_fixed_density_energy(ob, Pp))
            ob.prm[name][Z] = base
            w = (1.0, -8.0, 8.0, -1.0)
            col = COLUMNS.index(name)
            for k in (0, 1):
                d = sum(wk * e[k] for wk, e in zip(w, ev)) / (12 * h)
                g = np.bincount(mol[sel], weights=G[sel, k, col], minlength=ob.nmol)
                assert (np.abs(g - d) / (1.0 + np.abs(d))).max() < bar, (method, Z, name, k, g, d)


@pytest.mark.parametrize("method", ["MNDO", "AM1", "PM3"])
def test_param_grad_of_two_atom_systems(method):
    pairs = [(16, 8, 1.5), (17, 9, 1.7), (16, 16, 2.0), (17, 1, 1.35), (9, 1, 0.95), (1, 1, 0.8)]
    u = np.array([0.48, -0.6, 0.64])
    sp = np.array([p[:2] for p in pairs])
    c = np.array([[[0.0, 0.0, 0.0], p[2] * u] for p in pairs])
    _check(sp, c, method, 5, R.PARAM_NAMES[:12 + 3 * R.N_GAUSS[method]])


def test_param_grad_over_several_tiles():
    sp, c = W.alkanes(1, seed=9, nmin=9, nmax=9)  # 9 heavy atoms and 20 hydrogens
    _check(sp, c, "AM1", 6, ("zeta_s", "beta_p", "g_ss", "h_sp", "alpha", "Gaussian1_K"))
