"""The workgroup eigensolver on blocks whose levels are degenerate or nearly so, as those of symmetric molecules and of
identical molecules far apart are: densities and eigenpairs against numpy's float64 eigh.

Bars, for levels of 1..40 eV and a gap of 5 eV or more: a backward-stable solver's density is off by n eps |F| / gap,
below 4e-13 here, so 1e-12; vectors come out orthogonal to eps |T| over the solver's cluster
distance of 1e-3 |T|, 2e-13 and a small factor, so 5e-12, and with residuals of the size of eps times
|F|, so 1e-12 |F|.
"""
import numpy as np
import pytest
import torch

from pyseqm_amd.engine import SCFEngine
from pyseqm_amd.layout import PackedBatch

pytestmark = pytest.mark.gpu


def _spectrum(rng, n):
    o = n // 2
    return np.concatenate([-np.sort(rng.uniform(10.0, 40.0, o)), np.sort(rng.uniform(1.0, 20.0, n - o))])


def _with_levels(rng, lam):
    q, _ = np.linalg.qr(rng.normal(size=(len(lam), len(lam))))
    f = (q * lam) @ q.T
    return 0.5 * (f + f.T)


def _pairs(x):
    x[1::2] = x[0:len(x) - len(x) % 2:2]


def _block(rng, kind, n):
    """(matrix, occupied orbitals)"""
    lam, o = _spectrum(rng, n), n // 2
    if kind == "pairs":
        _pairs(lam[:o])
        _pairs(lam[o:])
    elif kind == "fours":
        lam[:o] = lam[0] + np.sort(rng.integers(0, max(o // 4, 1), o))
        lam[:o] -= lam[:o].max() + 5.0
    if kind in ("pairs", "fours"):
        return _with_levels(rng, lam), o
    # identical fragments with a weak coupling, orbitals in any order
    parts, coupling = {"two": (2, 1e-14), "four": (4, 0.0), "two coupled": (2, 1e-10)}[kind]
    h = n // parts
    f = np.kron(np.eye(parts), _with_levels(rng, _spectrum(rng, h)))
    for a in range(parts):
        for b in range(a):
            m = coupling * rng.normal(size=(h, h))
            f[a * h:a * h + h, b * h:b * h + h] = m
            f[b * h:b * h + h, a * h:a * h + h] = m.T
    p = rng.permutation(parts * h)
    return f[np.ix_(p, p)], parts * (h // 2)


@pytest.mark.parametrize("kind", ["pairs", "fours", "two", "four", "two coupled"])
@pytest.mark.parametrize("top", [48, 96, 138, 192])
def test_degenerate_levels(kind, top):
    rng = np.random.default_rng(top)
    blocks = [_block(rng, kind, n) for n in (top, top - 4, top // 2 + 2, 12) for _ in range(3)]
    norb = [len(f) for f, _ in blocks]
    nh = [n // 4 for n in norb]
    nH = [n - 4 * k for n, k in zip(norb, nh)]
    b = PackedBatch.from_counts(nh, nH, [o for _, o in blocks], max(x + y for x, y in zip(nh, nH)), "cuda")
    eng = SCFEngine(None, None, "AM1", "cuda", batch=b)
    F = torch.as_tensor(np.concatenate([f.reshape(-1) for f, _ in blocks]), device="cuda")
    P = torch.full_like(F, float("nan"))
    eng._idx_host = np.arange(len(norb))
    eng.density_eigh(F, torch.arange(len(norb), dtype=torch.int32, device="cuda"), len(norb), P)
    e, V = (t.cpu().numpy() for t in eng.eig(F))
    assert int(eng.eigh_fail.item()) == 0
    at = 0
    for k, (f, o) in enumerate(blocks):
        n = len(f)
        p = P[at:at + n * n].view(n, n).cpu().numpy()
        at += n * n
        w, U = np.linalg.eigh(f)
        scale = np.abs(w).max()
        assert np.abs(p - 2.0 * U[:, :o] @ U[:, :o].T).max() < 1e-12, n
        q, ev = V[k, :n, :n], e[k, :n]
        assert np.abs(np.sort(ev) - w).max() < 1e-12 * scale, n
        assert np.abs(q.T @ q - np.eye(n)).max() < 5e-12, n
        assert np.abs(f @ q - q * ev).max() < 1e-12 * scale, n
