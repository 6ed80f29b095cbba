"""pyseqm_eigh_density_large over its whole range of sizes, the smallest included, called directly: the densities
(levels, gap and bound of test_gpu_eigh_sizes.py), and nothing written behind its scratch."""
import numpy as np
import pytest
import torch

from pyseqm_amd import _native as nat
from pyseqm_amd.layout import PackedBatch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nmax", [1, 2, 3, 15, 16, 17, 31, 32, 47, 48, 49, 96, 97, 192])
def test_every_size(nmax):
    batch = [(n, o) for n in sorted({nmax, max(nmax - 1, 1), (nmax + 1) // 2, 1}, reverse=True) for o in {n, n // 2, 0}]
    nh = [n // 4 for n, _ in batch]
    nH = [n - 4 * k for (n, _), k in zip(batch, nh)]
    b = PackedBatch.from_counts(nh, nH, [o for _, o in batch], max(x + y for x, y in zip(nh, nH)), "cuda")
    rng = np.random.default_rng(nmax)
    fs, refs = [], []
    for n, o in batch:
        lam = np.concatenate([rng.uniform(-40.0, -10.0, o), rng.uniform(1.0, 20.0, n - o)])
        q, _ = np.linalg.qr(rng.normal(size=(n, n)))
        f = (q * lam) @ q.T
        fs.append(0.5 * (f + f.T))
        refs.append(2.0 * q[:, :o] @ q[:, :o].T)
    F = torch.as_tensor(np.concatenate([f.reshape(-1) for f in fs]), device="cuda")
    P = torch.full_like(F, float("nan"))
    idx = torch.arange(len(batch), dtype=torch.int32, device="cuda")
    size, guard = len(batch) * nmax * nmax, 4096
    ws, Z = (torch.full((k * size + guard,), -7.0, dtype=torch.float64, device="cuda") for k in (4, 1))
    fail = torch.zeros(1, dtype=torch.int32, device="cuda")
    nat.call("pyseqm_eigh_density_large", b.L, nat.ptr(idx), len(batch), nmax, nat.ptr(F), nat.ptr(P), nat.ptr(ws),
             nat.ptr(Z), nat.ptr(fail), nat.stream_ptr())
    torch.cuda.synchronize()
    assert bool((ws[4 * size:] == -7.0).all()) and bool((Z[size:] == -7.0).all())
    at = 0
    for (n, o), ref in zip(batch, refs):
        p = P[at:at + n * n].view(n, n).cpu().numpy()
        at += n * n
        assert np.array_equal(p, p.T), (n, o)
        assert np.abs(p - ref).max() < 1e-10, (n, o)
    assert int(fail.item()) == 0
