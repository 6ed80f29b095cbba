"""SCFEngine.eig's routes for batches that the all-eigenpairs solver takes in two launches (more than 256 blocks, some
above 139 orbitals).  On the CPU: the scratch of every launch is large enough and shares no memory with an output.  On
the GPU: energies and vectors against numpy's float64 eigh, reruns bitwise equal.

Bars: energies within 1e-10 of the block's scale, residual and orthogonality below 1e-9 of it, those of
test_gpu_eigh_sizes.py.
"""
import types

import numpy as np
import pytest
import torch

from pyseqm_amd import _native as nat
from pyseqm_amd import engine as eng_mod
from pyseqm_amd.engine import SCFEngine

BATCHES = {
    "one small block first": [14] + [146] * 300,
    "one small block last": [146] * 300 + [14],
    "one middle block": [182] * 300 + [62],
    "many small blocks": [182] * 300 + [14] * 50,
    "two large blocks": [128] * 1400 + [140] * 2,
}


@pytest.mark.parametrize("name", sorted(BATCHES))
def test_scratch_is_its_own(name, monkeypatch):
    norb = np.array(BATCHES[name])
    off = np.concatenate([[0], np.cumsum(norb)[:-1]])
    launches = []

    def call(entry, layout, *args):
        if entry == "pyseqm_eigh_vectors":
            _, count, top, _, _, evals, Q, ws, _, _ = args
            launches.append((count, top, evals, Q, ws))

    monkeypatch.setattr(nat, "call", call)
    monkeypatch.setattr(nat, "ptr", lambda t: t)  # the stand-in takes the tensors themselves
    eng = SCFEngine.__new__(SCFEngine)
    eng.device, eng.stream = torch.device("cpu"), None
    nmax = int(norb.max())
    eng.b = types.SimpleNamespace(norb=norb, nmol=len(norb), nmax=nmax, molsize=(nmax + 3) // 4, total=1, L=None)
    eng.orb_off = torch.as_tensor(off)
    monkeypatch.setattr(eng_mod.torch, "empty", _no_storage(torch.empty))
    eng.eig(torch.empty(1, dtype=torch.float64))
    assert len(launches) == 2 and sum(n for n, *_ in launches) == len(norb)
    for count, top, evals, Q, ws in launches:
        assert ws.numel() >= 4 * count * top ** 2
        assert ws.data_ptr() not in (evals.data_ptr(), Q.data_ptr())


def _no_storage(empty):
    """torch.empty whose large results take no memory: distinct one-element storages, expanded."""
    def f(*shape, **kw):
        shape = shape[0] if len(shape) == 1 and not isinstance(shape[0], int) else shape
        if int(np.prod(shape)) > 1 << 20:
            return empty(1, **kw).expand(*shape)
        return empty(*shape, **kw)
    return f


@pytest.mark.gpu
@pytest.mark.parametrize("name", sorted(BATCHES))
def test_eig_of_two_launches(name):
    from pyseqm_amd.layout import PackedBatch
    norb = BATCHES[name]
    nh = [n // 4 for n in norb]
    nH = [n - 4 * k for n, k in zip(norb, nh)]
    b = PackedBatch.from_counts(nh, nH, [n // 2 for n in norb], max(a + c for a, c in zip(nh, nH)), "cuda")
    eng = SCFEngine(None, None, "AM1", "cuda", batch=b)
    rng = np.random.default_rng(len(norb) + norb[0])
    fs = []
    for n in norb:
        f = rng.normal(size=(n, n))
        fs.append(f + f.T)
    F = torch.as_tensor(np.concatenate([f.reshape(-1) for f in fs]), device="cuda")
    e, V = eng.eig(F)
    e2, V2 = eng.eig(F)
    assert torch.equal(e, e2) and torch.equal(V, V2)
    e, V = e.cpu().numpy(), V.cpu().numpy()
    for k, (f, n) in enumerate(zip(fs, norb)):
        scale = np.abs(f).max() * np.sqrt(n)
        q = V[k, :n, :n]
        assert np.abs(e[k, :n] - np.linalg.eigvalsh(f)).max() < 1e-10 * scale, (k, n)
        assert not e[k, n:].any(), (k, n)
        assert np.abs(q.T @ q - np.eye(n)).max() < 1e-9, (k, n)
        assert np.abs(f @ q - q * e[k, :n]).max() < 1e-9 * scale, (k, n)
