"""eig()'s orbital energies ascend, as those of the library's solver do, also where levels agree to rounding."""
import numpy as np
import pytest
import torch

from pyseqm_amd.engine import SCFEngine
from pyseqm_amd.layout import PackedBatch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("top", [14, 48, 96, 139, 192])
def test_energies_ascend(top):
    rng = np.random.default_rng(top)
    norb = [top, max(top // 2, 2), 1] * 4
    fs = []
    for n in norb:  # three levels
        q, _ = np.linalg.qr(rng.normal(size=(n, n)))
        f = (q * rng.choice([-30.0, -11.0, 5.0], n)) @ q.T
        fs.append(0.5 * (f + f.T))
    nh = [n // 4 for n in norb]
    nH = [n - 4 * k for n, k in zip(norb, nh)]
    b = PackedBatch.from_counts(nh, nH, [n // 2 for n in norb], max(x + y for x, y in zip(nh, nH)), "cuda")
    eng = SCFEngine(None, None, "AM1", "cuda", batch=b)
    e, V = (t.cpu().numpy() for t in eng.eig(torch.as_tensor(np.concatenate([f.reshape(-1) for f in fs]), device="cuda")))
    for k, (f, n) in enumerate(zip(fs, norb)):
        assert (np.diff(e[k, :n]) >= 0.0).all(), (k, n)
        assert np.abs(e[k, :n] - np.linalg.eigvalsh(f)).max() < 1e-12 * 30.0, (k, n)
