"""The FP64 density step where a launch asks for all of a compute unit's LDS: the largest occupations that the size rule
(pyseqm_eigh_density_lds_ok) accepts at each block size, in one molecule and as the largest block of one
and the highest occupation of another; all eigenpairs at their limit in LDS.

Bars: densities and eigenpairs as in test_gpu_eigh_sizes.py, for the same levels and gap.
"""
import numpy as np
import pytest
import torch

from pyseqm_amd.engine import SCFEngine, eigh_wg_ok
from pyseqm_amd.layout import PackedBatch

pytestmark = pytest.mark.gpu


def _most(n):
    return max(o for o in range(n + 1) if eigh_wg_ok(n, o))


def _check(batch):
    nh = [n // 4 for n, _ in batch]
    nH = [n - 4 * k for (n, _), k in zip(batch, nh)]
    b = PackedBatch.from_counts(nh, nH, [o for _, o in batch], max(x + y for x, y in zip(nh, nH)), "cuda")
    eng = SCFEngine(None, None, "AM1", "cuda", batch=b)
    rng = np.random.default_rng(batch[0])
    fs, refs = [], []
    for n, o in batch:
        lam = np.concatenate([rng.uniform(-40.0, -10.0, o), rng.uniform(1.0, 20.0, n - o)])
        q, _ = np.linalg.qr(rng.normal(size=(n, n)))
        f = (q * lam) @ q.T
        fs.append(0.5 * (f + f.T))
        refs.append(2.0 * q[:, :o] @ q[:, :o].T)
    F = torch.as_tensor(np.concatenate([f.reshape(-1) for f in fs]), device="cuda")
    P = torch.full_like(F, float("nan"))
    eng._eigh_wg(F, np.arange(len(batch)), P)
    torch.cuda.synchronize()
    at = 0
    for (n, o), ref in zip(batch, refs):
        p = P[at:at + n * n].view(n, n).cpu().numpy()
        at += n * n
        assert np.array_equal(p, p.T), (n, o)
        assert np.abs(p - ref).max() < 1e-10, (n, o)
    assert int(eng.eigh_fail.item()) == 0


@pytest.mark.parametrize("n", [48, 96, 97, 139, 140, 169, 175, 178, 181, 182, 184, 188, 191, 192])
def test_highest_occupation(n):
    _check([(n, _most(n))])


@pytest.mark.parametrize("n", [169, 178, 184, 191, 192])
def test_largest_block_and_highest_occupation_of_two_molecules(n):
    o = _most(n)
    _check([(n, n // 3), (o + 30, o), (7, 3)])


def test_all_eigenpairs_at_the_limit():
    b = PackedBatch.from_counts([34], [3], [60], 40, "cuda")  # 139 orbitals
    eng = SCFEngine(None, None, "AM1", "cuda", batch=b)
    f = np.random.default_rng(3).normal(size=(139, 139))
    f = f + f.T
    e, V = (t.cpu().numpy()[0] for t in eng.eig(torch.as_tensor(f.reshape(-1), device="cuda")))
    scale = np.abs(f).max() * np.sqrt(139)
    assert np.abs(e[:139] - np.linalg.eigvalsh(f)).max() < 1e-10 * scale
    assert np.abs(V.T @ V - np.eye(139)).max() < 1e-9
