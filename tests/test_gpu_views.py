"""The view kernels (padded matrices, block array, dense integrals, pair indices, orbital charges) against the
index arrays of the host layout, element for element, over ragged batches: one atom, hydrogens only, heavy atoms
only, tile edges of 8 atoms.  They move values without arithmetic (charges: four squares, 1e-15)."""
import numpy as np
import pytest
import torch

from pyseqm_amd.engine import SCFEngine
from pyseqm_amd.layout import PackedBatch

pytestmark = pytest.mark.gpu
DEV = "cuda"
SHAPES = {"one atom": [(1, 0)], "hydrogens": [(0, 2), (0, 9)], "heavy": [(2, 0), (9, 0)],
          "ragged": [(1, 4), (8, 8), (9, 17), (0, 2), (7, 1), (16, 34), (1, 0)]}


def _batch(shapes):
    width = max(a + b for a, b in shapes)
    sp = np.zeros((len(shapes), width), dtype=np.int64)
    for m, (a, h) in enumerate(shapes):
        sp[m, :a] = 6
        sp[m, a:a + h] = 1
    charges = np.array([(4 * a + h) % 2 for a, h in shapes])
    return sp, PackedBatch(sp, "AM1", DEV, charges), PackedBatch(sp, "AM1", "cpu", charges)


@pytest.mark.parametrize("name", sorted(SHAPES))
def test_views_match_the_index_arrays(name):
    sp, b, host = _batch(SHAPES[name])
    rng = np.random.default_rng(3)
    x = rng.normal(size=b.total)
    X = torch.as_tensor(x, device=DEV)
    ref = host.to_padded(torch.as_tensor(x)).numpy()
    w = 4 * b.molsize
    assert np.array_equal(b.to_padded(X).cpu().numpy(), ref)
    assert np.array_equal(b.to_padded_upper(X).cpu().numpy(), np.triu(ref))
    blocks = np.triu(ref).reshape(b.nmol, b.molsize, 4, b.molsize, 4).transpose(0, 1, 3, 2, 4).reshape(-1, 4, 4)
    assert np.array_equal(b.to_blocks(X).cpu().numpy(), blocks)
    xp = rng.normal(size=(b.nmol, w, w))
    full = torch.as_tensor(xp, device=DEV)
    want = host.from_padded(torch.as_tensor(xp)).numpy()
    assert np.array_equal(b.from_padded(full).cpu().numpy(), want)
    assert np.array_equal(b.from_padded(full.transpose(1, 2).contiguous().transpose(1, 2)).cpu().numpy(), want)
    tracked = full.clone().requires_grad_(True)  # autograd still passes through
    assert torch.autograd.grad(b.from_padded(tracked).sum(), tracked)[0].sum() == b.total
    assert b.to_padded(X.float()).dtype == torch.float32
    assert np.array_equal(b.pair_ref_device()[:64 * b.ntiles].cpu().numpy(), host.pair_ref_host)


@pytest.mark.parametrize("name", sorted(SHAPES))
def test_dense_integrals_and_charges(name):
    sp, b, host = _batch(SHAPES[name])
    eng = SCFEngine(sp, None, "AM1", DEV, batch=b)
    rng = np.random.default_rng(4)
    want = np.zeros((b.npairs, 10, 10))
    for kind, buf in enumerate((eng.w_xx, eng.w_xh, eng.w_hh)):
        v = rng.normal(size=buf.numel())
        buf.copy_(torch.as_tensor(v))
        ref, idx = host.w_gather_index(kind, "cpu")
        if ref is not None:
            rows, ref = v[idx.numpy()], ref.numpy()
            if kind == 0:
                want[ref] = rows.reshape(-1, 10, 10)
            elif kind == 1:
                want[ref, :, 0] = rows
            else:
                want[ref, 0, 0] = rows[:, 0]
    assert np.array_equal(eng.w_reference().cpu().numpy(), want)
    V = torch.as_tensor(rng.normal(size=(b.nmol, b.nmax, b.nmax)), device=DEV)
    for v in (V, V.transpose(1, 2)):  # rows or columns contiguous
        v2 = v.cpu().numpy() ** 2
        want = np.zeros((b.nmol, 4 * b.molsize, b.molsize))
        for m in range(b.nmol):
            nh, nH = int(b.nheavy[m]), int(b.nhydro[m])
            n = 4 * nh + nH
            want[m, :n, :nh] = v2[m][:n, :4 * nh].reshape(n, 4, nh).sum(1)
            want[m, :n, nh:nh + nH] = v2[m][:n, 4 * nh:n]
        np.testing.assert_allclose(eng.orbital_charges(v).cpu().numpy(), want, rtol=1e-14, atol=0)
