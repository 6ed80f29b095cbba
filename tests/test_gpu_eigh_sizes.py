"""The workgroup eigensolver at the edges of its register grids (48, 96, 192 rows), of its 16-wide panels and
of its occupations, against numpy's float64 eigh.

Bars: the density within 1e-10 of the reference's (levels of 1..40 eV and a gap of 11 eV: n eps |F| / gap < 1e-12,
and eps |F| / gap < 1e-11 between levels of the nearest spacing drawn), exactly symmetric; eigenpairs
with residual and orthogonality below 1e-9 |F| (clusters are orthogonalised as a set); reruns bitwise equal.
"""
import numpy as np
import pytest
import torch

from pyseqm_amd.engine import SCFEngine, eigh_wg_ok
from pyseqm_amd.layout import PackedBatch

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _blocks(sizes, noccs, kind, seed):
    rng = np.random.default_rng(seed)
    out = []
    for n, o in zip(sizes, noccs):
        lam = np.concatenate([-np.sort(rng.uniform(10.0, 40.0, o)), np.sort(rng.uniform(1.0, 20.0, n - o))])
        if kind == "degenerate":  # pairs of equal levels
            for i in range(1, o, 2):
                lam[i] = lam[i - 1]
        elif kind == "close":  # clusters: spacings of 1e-6, 1e-9 and 1e-12 of the spectrum's width
            for i in range(1, o):
                if i % 7 < 3:
                    lam[i] = lam[i - 1] + (4e-5, 4e-8, 4e-11)[i % 7]
        Q, _ = np.linalg.qr(rng.normal(size=(n, n)))
        f = (Q * lam) @ Q.T
        if kind == "diagonal":
            f = np.diag(rng.permutation(lam))
        elif kind == "blocks":  # two decoupled halves
            f[:n // 2, n // 2:] = 0.0
            f[n // 2:, :n // 2] = 0.0
            f[np.arange(n), np.arange(n)] -= 30.0 * (np.arange(n) < o)
        out.append(0.5 * (f + f.T))
    return out


def _engine(sizes, noccs):
    nh = [n // 4 for n in sizes]
    nH = [n - 4 * k for n, k in zip(sizes, nh)]
    molsize = max(a + b for a, b in zip(nh, nH))
    b = PackedBatch.from_counts(nh, nH, noccs, molsize, DEV)
    return SCFEngine(None, None, "AM1", DEV, batch=b)


SETS = {48: [1, 2, 3, 4, 15, 16, 17, 31, 33, 47, 48], 96: [1, 3, 16, 49, 50, 64, 65, 80, 95, 96],
        192: [1, 2, 5, 97, 98, 112, 113, 128, 129, 160, 161, 182, 191, 192]}


@pytest.mark.parametrize("grid", sorted(SETS))
@pytest.mark.parametrize("kind", ["spread", "degenerate", "close", "diagonal", "blocks"])
def test_density_at_grid_edges(grid, kind):
    sizes = SETS[grid]
    noccs = [min([n // 2, n, 0, (2 * n) // 3, 1][k % 5] if n < 97 else n // 2 - k % 3, n) for k, n in enumerate(sizes)]
    eng = _engine(sizes, noccs)
    assert eigh_wg_ok(max(sizes), max(noccs))
    fs = _blocks(sizes, noccs, kind, grid)
    F = torch.as_tensor(np.concatenate([f.reshape(-1) for f in fs]), device=DEV)
    Ps = []
    for _ in range(2):
        P = torch.full_like(F, float("nan"))
        eng._eigh_wg(F, np.arange(len(sizes)), P)
        Ps.append(P)
    torch.cuda.synchronize()
    assert torch.equal(*Ps)
    o = 0
    for f, n, nocc in zip(fs, sizes, noccs):
        p = P[o:o + n * n].view(n, n).cpu().numpy()
        o += n * n
        w, U = np.linalg.eigh(f)
        if 0 < nocc < n and w[nocc] - w[nocc - 1] < 1.0:
            continue  # no gap in this block: its density is undetermined
        ref = 2.0 * U[:, :nocc] @ U[:, :nocc].T
        assert np.array_equal(p, p.T), n
        assert np.abs(p - ref).max() < 1e-10, (n, nocc, np.abs(p - ref).max())
    assert int(eng.eigh_fail.item()) == 0


@pytest.mark.parametrize("grid", sorted(SETS))
@pytest.mark.parametrize("kind", ["spread", "degenerate", "close", "diagonal"])
def test_eigenpairs_at_grid_edges(grid, kind):
    sizes = [n for n in SETS[grid] + [139] if n <= min(grid, 139)]
    eng = _engine(sizes, [n // 2 for n in sizes])
    fs = _blocks(sizes, [n // 2 for n in sizes], kind, grid + 1)
    F = torch.as_tensor(np.concatenate([f.reshape(-1) for f in fs]), device=DEV)
    Q = torch.full_like(F, float("nan"))
    off = np.concatenate([[0], np.cumsum(sizes)])
    evals = torch.full((int(off[-1]),), float("nan"), dtype=torch.float64, device=DEV)
    ws = torch.empty(4 * len(sizes) * max(sizes) ** 2, dtype=torch.float64, device=DEV)
    fail = torch.zeros(1, dtype=torch.int32, device=DEV)
    orb_off = torch.as_tensor(off[:-1].astype(np.int64), device=DEV)
    eng.eigenpairs(F, orb_off, evals, Q, ws, fail)
    torch.cuda.synchronize()
    o = 0
    for k, (f, n) in enumerate(zip(fs, sizes)):
        q = Q[o:o + n * n].view(n, n).cpu().numpy()
        o += n * n
        e = evals[int(off[k]):int(off[k]) + n].cpu().numpy()
        scale = np.abs(f).max() * np.sqrt(n)
        assert np.abs(e - np.linalg.eigvalsh(f)).max() < 1e-10 * scale, n
        assert np.abs(q.T @ q - np.eye(n)).max() < 1e-9, n
        assert np.abs(f @ q - q * e).max() < 1e-9 * scale, n
    assert int(fail.item()) == 0


@pytest.mark.parametrize("kind", ["spread", "degenerate", "close", "diagonal", "blocks"])
def test_eigenpairs_above_the_lds_limit(kind):
    """140 to 192 orbitals: the vectors stand in the output; blocks on both sides of the limit in one batch, and
    eig()'s padded view of the same pairs (the identity beyond a block, zero energies)."""
    sizes = [140, 5, 141, 159, 160, 139, 161, 182, 191, 192]
    eng = _engine(sizes, [n // 2 for n in sizes])
    fs = _blocks(sizes, [n // 2 for n in sizes], kind, 7)
    F = torch.as_tensor(np.concatenate([f.reshape(-1) for f in fs]), device=DEV)
    e, V = (t.cpu().numpy() for t in eng.eig(F))
    assert V.shape == (len(sizes), 192, 192) and e.shape == (len(sizes), 4 * eng.b.molsize)
    for k, (f, n) in enumerate(zip(fs, sizes)):
        scale = np.abs(f).max() * np.sqrt(n)
        want = np.eye(192)
        want[:n, :n] = V[k, :n, :n]
        q = V[k, :n, :n]
        assert np.array_equal(V[k], want) and not e[k, n:].any(), n
        assert np.abs(e[k, :n] - np.linalg.eigvalsh(f)).max() < 1e-10 * scale, n
        assert np.abs(q.T @ q - np.eye(n)).max() < 1e-9, n
        assert np.abs(f @ q - q * e[k, :n]).max() < 1e-9 * scale, n


@pytest.mark.parametrize("kind", ["spread", "degenerate", "close", "diagonal", "blocks"])
def test_density_with_vectors_in_memory(kind):
    """Blocks of up to 192 orbitals whose occupied vectors do not fit LDS, beside one that does, through the density step:
    the bound of test_density_at_grid_edges."""
    sizes, noccs = [168, 180, 40, 191, 192, 192, 175], [112, 120, 20, 191, 128, 192, 174]
    eng = _engine(sizes, noccs)
    assert eigh_wg_ok(sizes, noccs).tolist() == [n == 40 or n * o + 3 * n + 704 <= 20480 for n, o in zip(sizes, noccs)]
    fs = _blocks(sizes, noccs, kind, 11)
    F = torch.as_tensor(np.concatenate([f.reshape(-1) for f in fs]), device=DEV)
    P = torch.full_like(F, float("nan"))
    eng._idx_host = np.arange(len(sizes))
    eng.eigh_log.clear()
    eng.density_eigh(F, torch.arange(len(sizes), dtype=torch.int32, device=DEV), len(sizes), P)
    assert all(how == "workgroup" for _, _, how in eng.eigh_log)
    o = 0
    for f, n, nocc in zip(fs, sizes, noccs):
        p = P[o:o + n * n].view(n, n).cpu().numpy()
        o += n * n
        w, U = np.linalg.eigh(f)
        ref = 2.0 * U[:, :nocc] @ U[:, :nocc].T
        assert np.array_equal(p, p.T), n
        assert np.abs(p - ref).max() < 1e-10, (n, nocc, np.abs(p - ref).max())
    assert int(eng.eigh_fail.item()) == 0
