"""The density step on blocks of two decoupled halves (the tridiagonal form splits), over all three register grids, with a
gap between occupied and virtual levels by construction so that every block counts: bounds of
test_gpu_eigh_sizes.py, exact symmetry and bitwise reruns."""
import numpy as np
import pytest
import torch

from pyseqm_amd.engine import SCFEngine
from pyseqm_amd.layout import PackedBatch

pytestmark = pytest.mark.gpu
SETS = {48: [2, 3, 4, 15, 16, 17, 31, 33, 47, 48], 96: [3, 16, 49, 50, 64, 65, 80, 95, 96],
        192: [2, 5, 97, 98, 112, 113, 128, 129, 160, 161, 182, 191, 192]}


def _half(rng, n, o):
    lam = np.concatenate([rng.uniform(-40.0, -10.0, o), rng.uniform(1.0, 20.0, n - o)])
    q, _ = np.linalg.qr(rng.normal(size=(n, n)))
    f = (q * lam) @ q.T
    return 0.5 * (f + f.T), 2.0 * q[:, :o] @ q[:, :o].T


@pytest.mark.parametrize("grid", sorted(SETS))
@pytest.mark.parametrize("shuffled", [False, True])
def test_two_halves(grid, shuffled):
    rng = np.random.default_rng(grid)
    fs, refs, noccs = [], [], []
    for k, n in enumerate(SETS[grid]):
        h = n // 2
        # occupied orbitals of the halves: half, all and none, a third
        o1, o2 = [(h // 2, (n - h) // 2), (h, 0), (h // 3, (n - h) // 2)][k % 3]
        (a, pa), (b, pb) = _half(rng, h, o1), _half(rng, n - h, o2)
        f, p = (np.block([[x, np.zeros((h, n - h))], [np.zeros((n - h, h)), y]]) for x, y in ((a, b), (pa, pb)))
        at = rng.permutation(n) if shuffled else np.arange(n)
        fs.append(f[np.ix_(at, at)])
        refs.append(p[np.ix_(at, at)])
        noccs.append(o1 + o2)
    nh = [n // 4 for n in SETS[grid]]
    nH = [n - 4 * k for n, k in zip(SETS[grid], nh)]
    batch = PackedBatch.from_counts(nh, nH, noccs, max(x + y for x, y in zip(nh, nH)), "cuda")
    eng = SCFEngine(None, None, "AM1", "cuda", batch=batch)
    F = torch.as_tensor(np.concatenate([f.reshape(-1) for f in fs]), device="cuda")
    out = []
    for _ in range(2):
        P = torch.full_like(F, float("nan"))
        eng._eigh_wg(F, np.arange(len(fs)), P)
        out.append(P.cpu().numpy())
    assert np.array_equal(*out) and int(eng.eigh_fail.item()) == 0
    at = 0
    for n, ref in zip(SETS[grid], refs):
        p = out[0][at:at + n * n].reshape(n, n)
        at += n * n
        assert np.array_equal(p, p.T), n
        assert np.abs(p - ref).max() < 1e-10, n
