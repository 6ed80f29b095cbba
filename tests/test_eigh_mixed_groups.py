"""The FP64 density step on batches whose largest block and highest occupation belong to different molecules: each block
fits the workgroup eigensolver's LDS, a launch sized by both does not.  On the CPU: every launch is within the
library's size rule and every block in exactly one.  On the GPU: the densities, with the bound of
test_gpu_eigh_sizes.py (levels and gap as there).
"""
import types

import numpy as np
import pytest
import torch

from pyseqm_amd import _native as nat
from pyseqm_amd.engine import SCFEngine, eigh_wg_ok

# (orbitals, occupied): an alkane of 30 carbons with 27 waters, and more of either side of the limits
BATCHES = [
    [(182, 91), (162, 108)],
    [(192, 96), (162, 108), (150, 100), (40, 20), (156, 104)],
    [(139, 139), (192, 1), (48, 48)],
    [(182, 91), (192, 128), (162, 108), (14, 7)],  # one whose vectors never fit
    [(182, 91), (156, 104), (8, 4)],               # fits as it is
]


@pytest.mark.parametrize("batch", BATCHES)
def test_launches_fit(batch, monkeypatch):
    norb, nocc = (np.array(x) for x in zip(*batch))
    lib = nat.lib()
    eng = SCFEngine.__new__(SCFEngine)
    eng.device, eng.stream = torch.device("cpu"), None
    eng.b = types.SimpleNamespace(norb=norb, nocc=nocc, nmol=len(norb))
    seen = []

    def run(F, idx, count, nmax, nocc_max, Pout, large=False):
        ids = idx.numpy()
        assert count == len(ids) and nmax == norb[ids].max() and nocc_max == nocc[ids].max()
        assert large or lib.pyseqm_eigh_density_lds_ok(nmax, nocc_max), (nmax, nocc_max)
        seen.extend(ids.tolist())

    monkeypatch.setattr(eng, "_eigh_wg_run", run, raising=False)
    eng._idx_host = np.arange(len(norb))
    assert eng.density_eigh(None, None, len(norb), None) is None
    assert sorted(seen) == list(range(len(norb)))
    whole = eng._eigh_wg_list(np.arange(len(norb)))
    assert (whole is not None) == bool(eigh_wg_ok(norb.max(), nocc.max()))


@pytest.mark.gpu
@pytest.mark.parametrize("batch", BATCHES)
def test_density(batch):
    from pyseqm_amd.layout import PackedBatch
    nh = [n // 4 for n, _ in batch]
    nH = [n - 4 * k for (n, _), k in zip(batch, nh)]
    b = PackedBatch.from_counts(nh, nH, [o for _, o in batch], max(x + y for x, y in zip(nh, nH)), "cuda")
    eng = SCFEngine(None, None, "AM1", "cuda", batch=b)
    rng = np.random.default_rng(len(batch))
    fs, refs = [], []
    for n, o in batch:
        lam = np.concatenate([rng.uniform(-40.0, -10.0, o), rng.uniform(1.0, 20.0, n - o)])
        q, _ = np.linalg.qr(rng.normal(size=(n, n)))
        f = (q * lam) @ q.T
        fs.append(0.5 * (f + f.T))
        refs.append(2.0 * q[:, :o] @ q[:, :o].T)
    F = torch.as_tensor(np.concatenate([f.reshape(-1) for f in fs]), device="cuda")
    P = torch.full_like(F, float("nan"))
    eng._idx_host = np.arange(len(batch))
    eng.density_eigh(F, torch.arange(len(batch), dtype=torch.int32, device="cuda"), len(batch), P)
    assert all(how == "workgroup" for _, _, how in eng.eigh_log)
    at = 0
    for (n, o), ref in zip(batch, refs):
        p = P[at:at + n * n].view(n, n).cpu().numpy()
        at += n * n
        assert np.array_equal(p, p.T), (n, o)
        assert np.abs(p - ref).max() < 1e-10, (n, o)
    assert int(eng.eigh_fail.item()) == 0
