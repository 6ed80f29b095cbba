"""The Krylov step's kernels (pyseqm_krylov_start / response / fit / combine) and the tiled Fermi density against
float64 numpy: blocks over the 16-orbital tile edges, ranks up to the largest, the largest block whose response takes one
launch, and the product path beside it."""
import numpy as np
import pytest
import torch

from pyseqm_amd import _native as nat
from pyseqm_amd import ksa as K
from pyseqm_amd.engine import SCFEngine
from pyseqm_amd.layout import PackedBatch

pytestmark = pytest.mark.gpu
DEV = "cuda"
SIZES = {"edges": [2, 3, 15, 16, 17, 31, 33, 48, 49], "largest": [78, 64, 65, 5], "products": [79, 112, 20]}


def _setup(name, rank):
    sizes = SIZES[name]
    nh = [n // 4 for n in sizes]
    nH = [n - 4 * k for n, k in zip(sizes, nh)]
    b = PackedBatch.from_counts(nh, nH, [max(1, n // 2) for n in sizes], max(a + c for a, c in zip(nh, nH)), DEV)
    eng = SCFEngine(None, None, "AM1", DEV, batch=b)
    return sizes, b, eng, K.KSAWorkspace(eng, rank)


def _blocks(b, t):
    t = t.cpu().numpy()
    return [t[int(o):int(o) + int(n) ** 2].reshape(int(n), int(n)) for o, n in zip(b.mol_mat_off, b.norb)]


def _sym(rng, sizes, scale=1.0):
    out = [scale * rng.normal(size=(n, n)) / np.sqrt(n) for n in sizes]
    return [0.5 * (x + x.T) for x in out]


def _pack(blocks):
    return torch.as_tensor(np.concatenate([x.reshape(-1) for x in blocks]), device=DEV)


@pytest.mark.parametrize("name", sorted(SIZES))
@pytest.mark.parametrize("rank", [1, 3, 8])
def test_krylov_vectors(name, rank):
    """Errors: a few n eps per product of blocks of unit norm (1e-12 here); the fit's system is compared, its
    solution against numpy's from the kernel's own system, relative to the condition it has."""
    sizes, b, eng, ks = _setup(name, rank)
    rank = min(rank, min(sizes) ** 2)
    rng = np.random.default_rng(rank)
    T, kT = 10000.0, K.KB_EV * 10000.0
    lam = [np.sort(rng.uniform(-30.0, 10.0, n)) for n in sizes]
    Qs = [np.linalg.qr(rng.normal(size=(n, n)))[0] for n in sizes]
    mus = [0.5 * (e[max(1, n // 2) - 1] + e[max(1, n // 2)]) for e, n in zip(lam, sizes)]
    ks.Q.copy_(_pack(Qs))
    ks.evals.copy_(torch.as_tensor(np.concatenate(lam)))
    ks.mu.copy_(torch.as_tensor(np.array(mus)))
    D, P = _sym(rng, sizes), _sym(rng, sizes)
    Dt, Pt = _pack(D), _pack(P)
    assert ks.fused == (name != "products")
    Vs, Ws = [], []
    for k in range(rank):
        nat.call("pyseqm_krylov_start", b.L, nat.ptr(ks.idx), b.nmol, k, nat.ptr(Dt), nat.ptr(Pt), nat.ptr(ks.dDS),
                 nat.ptr(ks.V), nat.ptr(ks.W), ks.V.stride(0), eng.stream)
        V = [(d - p) if k == 0 else w.copy() for d, p, w in zip(D, P, Ws[-1] if Ws else D)]
        for m in range(len(sizes)):
            for vj in Vs:
                V[m] = V[m] - (V[m] * vj[m]).sum() * vj[m]
            V[m] /= np.sqrt((V[m] ** 2).sum())
        got = _blocks(b, ks.V[k])
        # Gram-Schmidt loses |W| / |what is left|: compared where more than 1e-3 of the residual is left
        for m, n in enumerate(sizes):
            if k < n:
                assert np.abs(got[m] - V[m]).max() < 1e-9, (n, k)
        Vs.append(got)  # go on from the kernel's own vectors
        G = _sym(rng, sizes, 3.0)
        ks.G.copy_(_pack(G))
        K._response(eng, ks, k, T, K.KB_EV)
        W = _blocks(b, ks.W[k])
        for m, n in enumerate(sizes):
            beta = 1.0 / kT
            cn = beta * 2.0 ** (-2 - K.CANON_DM_PRT_ITER)
            p0 = 0.5 - cn * (lam[m] - mus[m])
            P1 = -cn * (Qs[m].T @ G[m] @ Qs[m])
            for _ in range(K.CANON_DM_PRT_ITER):
                dX = p0[:, None] * P1 + P1 * p0[None]
                iD = 1.0 / (2.0 * (p0 * p0 - p0) + 1.0)
                p0 = iD * p0 * p0
                P1 = iD[:, None] * (dX + 2.0 * (P1 - dX) * p0[None])
            dp = beta * p0 * (1.0 - p0)
            P1 = P1 + np.diag(dp) * (-np.trace(P1) / dp.sum())
            want = Qs[m] @ P1 @ Qs[m].T - got[m]
            assert np.abs(W[m] - want).max() < 1e-12 * max(1.0, np.abs(P1).max()) * n, (n, k)
        Ws.append(W)
        O, rhs, alpha = ks.O.cpu().numpy(), ks.rhs.cpu().numpy(), ks.alpha.cpu().numpy()
        for m, n in enumerate(sizes):
            w = np.stack([x[m].reshape(-1) for x in Ws])
            gram, r = w @ w.T, w @ (D[m] - P[m]).reshape(-1)
            assert np.abs(O[m, :k + 1, :k + 1] - gram).max() < 1e-12 * np.abs(gram).max() * n
            assert np.abs(rhs[m, :k + 1] - r).max() < 1e-12 * np.sqrt(np.abs(gram).max()) * n
            cond = np.linalg.cond(O[m, :k + 1, :k + 1])
            if cond < 1e10:
                a = np.linalg.solve(O[m, :k + 1, :k + 1], rhs[m, :k + 1])
                assert np.abs(alpha[m, :k + 1] - a).max() < 1e-14 * cond * max(1.0, np.abs(a).max()), (n, k)
    out = torch.empty_like(ks.G)
    nat.call("pyseqm_krylov_combine", b.L, nat.ptr(ks.idx), b.nmol, int(b.nmax), rank, nat.ptr(ks.alpha),
             nat.ptr(ks.V), ks.V.stride(0), nat.ptr(out), eng.stream)
    for m, x in enumerate(_blocks(b, out)):
        want = -sum(alpha[m, i] * Vs[i][m] for i in range(rank))
        assert np.abs(x - want).max() < 1e-13 * max(1.0, np.abs(alpha[m, :rank]).max()) * rank


@pytest.mark.parametrize("name", sorted(SIZES))
@pytest.mark.parametrize("T", [300.0, 10000.0])
def test_fermi_density_tiles(name, T):
    """mu to the recorded step's residual (1e-9 electrons), D = 2 Q f Q^T to n eps, bitwise symmetric."""
    sizes, b, eng, ks = _setup(name, 1)
    rng = np.random.default_rng(5)
    lam = [np.sort(rng.uniform(-30.0, 10.0, n)) for n in sizes]
    Qs = [np.linalg.qr(rng.normal(size=(n, n)))[0] for n in sizes]
    ks.Q.copy_(_pack(Qs))
    ks.evals.copy_(torch.as_tensor(np.concatenate(lam)))
    D = torch.full_like(ks.Q, float("nan"))
    nat.call("pyseqm_fermi_density", b.L, nat.ptr(ks.idx), b.nmol, int(b.nmax), nat.ptr(ks.orb_off), nat.ptr(ks.evals),
             nat.ptr(ks.Q), T, K.KB_EV, nat.ptr(ks.occ), nat.ptr(ks.mu), nat.ptr(D), nat.ptr(ks.S), nat.ptr(ks.work),
             eng.stream)
    mu, occ, S = ks.mu.cpu().numpy(), ks.occ.cpu().numpy(), ks.S.cpu().numpy()
    o = 0
    for m, (n, d) in enumerate(zip(sizes, _blocks(b, D))):
        with np.errstate(over="ignore"):
            f = 1.0 / (1.0 + np.exp((lam[m] - mu[m]) / (K.KB_EV * T)))
        assert np.abs(occ[o:o + n] - f).max() < 1e-13
        assert abs(occ[o:o + n].sum() - max(1, n // 2)) < 2e-9
        g = f[(f > 1e-14) & (1 - f > 1e-14)]
        assert abs(S[m] + K.KB_EV * (g * np.log(g) + (1 - g) * np.log(1 - g)).sum()) < 1e-13 * n
        assert np.array_equal(d, d.T)
        assert np.abs(d - 2.0 * (Qs[m] * f) @ Qs[m].T).max() < 1e-14 * n
        o += n
