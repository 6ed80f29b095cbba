"""The workgroup eigensolver on more blocks than run at once (where the variants for up to 48 and up to 96 orbitals are
held to two waves per SIMD), and on as many as do: every block's density and eigenpairs against numpy's, with the
bounds of test_gpu_eigh_sizes.py, plain and degenerate levels.
"""
import numpy as np
import pytest
import torch

from pyseqm_amd.engine import SCFEngine
from pyseqm_amd.layout import PackedBatch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("sizes,count", [([48, 33, 16, 8, 1], 1024), ([48, 33, 16, 8, 1], 1025), ([8, 4], 1500),
                                         ([96, 65, 49, 20], 256), ([96, 65, 49, 20], 257)])
def test_many_blocks(sizes, count):
    rng = np.random.default_rng(count)
    kinds = []
    for n in sizes:
        for pairs in (False, True):
            o = n // 2
            lam = np.concatenate([rng.uniform(-40.0, -10.0, o), rng.uniform(1.0, 20.0, n - o)])
            if pairs:
                lam[1:o:2] = lam[0:o - o % 2:2]
            q, _ = np.linalg.qr(rng.normal(size=(n, n)))
            f = (q * lam) @ q.T
            f = 0.5 * (f + f.T)
            w, U = np.linalg.eigh(f)
            kinds.append((f, o, 2.0 * U[:, :o] @ U[:, :o].T, w))
    pick = [kinds[k % len(kinds)] for k in range(count)]
    norb = [len(f) for f, *_ in pick]
    nh = [n // 4 for n in norb]
    nH = [n - 4 * k for n, k in zip(norb, nh)]
    b = PackedBatch.from_counts(nh, nH, [o for _, o, *_ in pick], max(x + y for x, y in zip(nh, nH)), "cuda")
    eng = SCFEngine(None, None, "AM1", "cuda", batch=b)
    F = torch.as_tensor(np.concatenate([f.reshape(-1) for f, *_ in pick]), device="cuda")
    P = torch.full_like(F, float("nan"))
    eng._idx_host = np.arange(count)
    eng.density_eigh(F, torch.arange(count, dtype=torch.int32, device="cuda"), count, P)
    e, V = (t.cpu().numpy() for t in eng.eig(F))
    P = P.cpu().numpy()
    assert int(eng.eigh_fail.item()) == 0
    at = 0
    for k, (f, o, ref, w) in enumerate(pick):
        n = len(f)
        p = P[at:at + n * n].reshape(n, n)
        at += n * n
        assert np.array_equal(p, p.T) and np.abs(p - ref).max() < 1e-10, (k, n)
        q, scale = V[k, :n, :n], np.abs(f).max() * np.sqrt(n)
        assert np.abs(e[k, :n] - w).max() < 1e-10 * scale, (k, n)
        assert np.abs(q.T @ q - np.eye(n)).max() < 1e-9, (k, n)
        assert np.abs(f @ q - q * e[k, :n]).max() < 1e-9 * scale, (k, n)
