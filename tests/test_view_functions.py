"""The module functions that take the reference's padded arrays as they are, on any device: the block array of a matrix
(the inverse of blocks_to_matrix) and the orbital charges (scf_loop.py:2376-2387), against loops."""
import types

import torch

from pyseqm_amd.seqm_functions.fock import blocks_to_matrix, matrix_to_blocks
from pyseqm_amd.seqm_functions.scf_loop import orbital_charges


def test_matrix_to_blocks():
    nmol, m = 3, 5
    X = torch.randn(nmol, 4 * m, 4 * m, dtype=torch.float64, generator=torch.Generator().manual_seed(1))
    X = X + X.transpose(1, 2)
    M = matrix_to_blocks(X, nmol, m)
    assert M.shape == (nmol * m * m, 4, 4)
    for k in range(nmol):
        for i in range(m):
            for j in range(m):
                want = X[k].triu()[4 * i:4 * i + 4, 4 * j:4 * j + 4]
                assert torch.equal(M[(k * m + i) * m + j], want)
    assert torch.equal(blocks_to_matrix(M, nmol, m), X)


def test_orbital_charges():
    nh, nH, m = [2, 1, 0], [3, 0, 2], 6
    n = [4 * a + b for a, b in zip(nh, nH)]
    mol = types.SimpleNamespace(nmol=3, molsize=m, nHeavy=torch.tensor(nh), nHydro=torch.tensor(nH))
    for dtype in (torch.float64, torch.float32):
        v = torch.randn(3, max(n), max(n), dtype=dtype, generator=torch.Generator().manual_seed(2))
        v.requires_grad_(True)
        q = orbital_charges(mol, v)
        assert q.shape == (3, 4 * m, m) and q.dtype == dtype
        want = torch.zeros(3, 4 * m, m, dtype=dtype)
        for k in range(3):
            for o in range(n[k]):
                for a in range(nh[k] + nH[k]):
                    cols = [c * nh[k] + a for c in range(4)] if a < nh[k] else [3 * nh[k] + a]
                    want[k, o, a] = sum(v[k, o, c].detach() ** 2 for c in cols)
        torch.testing.assert_close(q.detach(), want)
        q.sum().backward()
        assert v.grad is not None
