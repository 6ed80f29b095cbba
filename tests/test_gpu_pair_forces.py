"""The closed-form pair forces (k_pair_forces) against the oracle's finite differences, pair by pair.

Two-atom systems of every tile kind and row combination of the overlaps, at random symmetric densities, with
the pair axis in general position, along +x, along -x (inside the antipodal cone of the quaternion frame, where
a frame is constant) and 1e-3 rad off -x (outside it); and one molecule of each kind of tile edge.  The
oracle differentiates with a 1e-4 A step: rounding of its overlap recurrences (up to 1e-11 relative) over the
step is below 1e-6 eV/A, the bar.
"""
import numpy as np
import pytest
import torch

from oracle import seqm_ref as R
from pyseqm_amd import workloads as W
from pyseqm_amd.engine import SCFEngine

pytestmark = pytest.mark.gpu
DEV = "cuda"
AXES = {"general": (0.48, -0.6, 0.64), "+x": (1.0, 0.0, 0.0), "-x": (-1.0, 0.0, 0.0),
        "near -x": (-np.cos(1e-3), np.sin(1e-3), 0.0)}


def _random_density(eng, rng):
    P = torch.zeros_like(eng.H)
    for m in range(eng.b.nmol):
        n, o = int(eng.b.norb[m]), int(eng.b.mol_mat_off[m])
        a = 0.3 * rng.normal(size=(n, n))
        P[o:o + n * n] = torch.as_tensor((a + a.T + np.diag(rng.uniform(0.5, 1.5, n))).reshape(-1), device=DEV)
    return P


def _check(sp, x, method, seed):
    eng = SCFEngine(sp, x, method, DEV)
    b = eng.b
    rng = np.random.default_rng(seed)
    P, D = _random_density(eng, rng), _random_density(eng, rng)
    Pp, Dp = b.to_padded(P).cpu().numpy(), b.to_padded(D).cpu().numpy()
    f = b.atom_to_padded(eng.forces(P)).cpu().numpy()
    np.testing.assert_allclose(f, R.forces_fd(sp, x, method, Pp), atol=1e-6, rtol=0)
    from pyseqm_amd import _native as nat
    out = torch.zeros(b.natoms, 3, dtype=torch.float64, device=DEV)
    nat.call("pyseqm_pair_forces_xl", b.L, nat.METHODS[method], nat.ptr(eng.coords), nat.ptr(eng.atom_par),
             nat.ptr(D), nat.ptr(P), 1.0e-3, nat.ptr(eng.part), nat.ptr(out), eng.stream)
    np.testing.assert_allclose(b.atom_to_padded(out).cpu().numpy(), R.forces_fd(sp, x, method, Pp, D=Dp), atol=1e-6,
                               rtol=0)


@pytest.mark.parametrize("axis", sorted(AXES))
@pytest.mark.parametrize("method", ["MNDO", "AM1", "PM3"])
def test_pair_forces_of_two_atoms(method, axis):
    pairs = [(1, 1, 0.9), (8, 6, 1.2), (9, 1, 1.0), (17, 1, 1.4), (16, 8, 1.6), (17, 9, 1.7), (16, 16, 2.0),
             (6, 6, 3.5)]
    sp = np.array([p[:2] for p in pairs])
    u = np.array(AXES[axis])
    x = np.array([[[0.1, -0.2, 0.3], np.array([0.1, -0.2, 0.3]) + p[2] * u] for p in pairs])
    _check(sp, x, method, 3)


@pytest.mark.parametrize("n", [3, 9])
def test_pair_forces_at_tile_edges(n):
    """n heavy atoms and 2 n + 2 hydrogens: full, partly filled and missing 8 x 8 tiles."""
    sp, x = W.alkanes(1, seed=n, nmin=n, nmax=n)
    _check(sp, x, "AM1", n)
