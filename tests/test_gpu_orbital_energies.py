"""eig()'s orbital energies to rounding: against eigenvalues refined in extended precision, for random spectra and all
three register grids of the workgroup eigensolver.

Bar: 6e-16 of the spectrum's largest value.  That is the largest error that the library's batched solver, whose
place the workgroup eigensolver takes in eig(), showed on such blocks (3.0e-16 to 5.7e-16 over 14 to 192 orbitals).
"""
import numpy as np
import pytest
import torch

from pyseqm_amd.engine import SCFEngine
from pyseqm_amd.layout import PackedBatch

pytestmark = pytest.mark.gpu
LD = np.longdouble


def _refined(A):
    """Eigenvalues of a symmetric float64 matrix with simple, separated levels, in extended precision: its float64
    vectors orthonormalised and corrected to first order until they stand."""
    n = len(A)
    V, A, one = np.linalg.eigh(A)[1].astype(LD), A.astype(LD), np.eye(n, dtype=LD)
    for _ in range(3):
        for _ in range(2):
            V = V @ (LD(1.5) * one - LD(0.5) * (V.T @ V))
        B = V.T @ A @ V
        gap = np.diag(B)[None, :] - np.diag(B)[:, None]
        np.fill_diagonal(gap, 1)
        X = (B - np.diag(np.diag(B))) / gap
        V = V @ (one + X)
    V = V @ (LD(1.5) * one - LD(0.5) * (V.T @ V))
    return np.sort(np.diag(V.T @ A @ V))


@pytest.mark.parametrize("n", [14, 48, 96, 139, 140, 192])
def test_energies_to_rounding(n):
    rng = np.random.default_rng(n)
    fs = []
    for _ in range(2):
        lam = np.concatenate([np.linspace(-40.0, -10.0, n // 2), np.linspace(1.0, 20.0, n - n // 2)])
        lam += rng.uniform(-0.05, 0.05, n)
        q, _ = np.linalg.qr(rng.normal(size=(n, n)))
        f = (q * lam) @ q.T
        fs.append(0.5 * (f + f.T))
    nh = n // 4
    b = PackedBatch.from_counts([nh] * 2, [n - 4 * nh] * 2, [n // 2] * 2, n - 3 * nh, "cuda")
    eng = SCFEngine(None, None, "AM1", "cuda", batch=b)
    e, _ = eng.eig(torch.as_tensor(np.concatenate([f.reshape(-1) for f in fs]), device="cuda"))
    for k, f in enumerate(fs):
        w = _refined(f)
        err = np.abs(e[k, :n].cpu().numpy() - w).max() / np.abs(w).max()
        assert err < 6e-16, float(err)
