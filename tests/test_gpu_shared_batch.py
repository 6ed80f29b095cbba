"""One packed batch used from two streams: its pair references, made on the first stream's request while that
stream is busy, are whole for the second; per-pair core repulsions of two engines on streams of their own agree."""
import numpy as np
import pytest
import torch

from pyseqm_amd.engine import SCFEngine
from pyseqm_amd.layout import PackedBatch

pytestmark = pytest.mark.gpu


def test_pair_references_across_streams(xyz):
    sp, X = xyz(["methane.xyz", "benzene.xyz"])
    b = PackedBatch(sp, "AM1", torch.device("cuda"))
    first, second = torch.cuda.Stream(), torch.cuda.Stream()
    with torch.cuda.stream(first):
        torch.cuda._sleep(20_000_000)
        a = b.pair_ref_device()
    with torch.cuda.stream(second):
        got = b.pair_ref_device().clone()
    second.synchronize()
    assert got.data_ptr() != a.data_ptr()
    host = PackedBatch(sp, "AM1", torch.device("cpu"))
    assert np.array_equal(got.cpu().numpy()[:64 * b.ntiles], host.pair_ref_host)


def test_two_engines_on_two_streams(xyz):
    sp, X = xyz(["methane.xyz", "benzene.xyz"])
    dev = torch.device("cuda")
    b = PackedBatch(sp, "AM1", dev)
    out = []
    for _ in range(2):
        s = torch.cuda.Stream()
        with torch.cuda.stream(s):
            eng = SCFEngine(sp, None, "AM1", dev, batch=b)
            eng.set_coordinates(torch.as_tensor(X, device=dev), enuc_pair=True)
            out.append((eng.enuc_pair, eng.enuc))
    torch.cuda.synchronize()
    assert torch.equal(out[0][0], out[1][0])
    assert abs(float(out[0][0].sum() - out[0][1].sum())) < 1e-9 * float(out[0][1].sum())
