"""Device SCF engine: drives the gfx950 kernels of libpyseqm_hip.so on one packed batch.

Host code only schedules kernels and reads one byte per molecule per SCF iteration (the
convergence flags), like the reference's ``int(notconverged.sum())`` host sync
(seqm/seqm_functions/scf_loop.py:1101).  Every floating-point array lives on the device.
"""
import collections
import math
import warnings

import numpy as np
import torch

from . import _native as nat
from .layout import PackedBatch
from .seqm_functions.constants import EHEAT, GP2C, GPPC, GSPC, GSSC, HSPC, TORE, UPPC, USSC, ev_kcalpmol
from .seqm_functions.parameters import COLUMNS, param_table

MAX_ITER = 1000
NFOCK = 10
SP2_DIIS_TOL = 1.0e-2


class SCFResult:
    pass


# Batched FP64 eigensolves of blocks with n <= 64 take a far slower solver path than n >= 68
# (measured on MI355X with the ROCm 7 solver: 1024 blocks of 64 take 417 ms, of 68 take 8 ms), so
# a group of many small blocks is padded up to this size (on 1024 alkanes a floor of 32 or 48 made
# the FP64 SCF 2.3-2.9x slower, 96 or 128 3-33 % slower).
EIGH_MIN_N = 68
# the floor applies to batched solves of at least this many blocks (a handful of small blocks is
# solved unpadded; the slow small-block path only costs at batch scale)
EIGH_MIN_N_BATCH = 16
# largest block whose DIIS residual stays on the FP64 GEMM with the mixed-precision density (the
# bf16x3 commutator is faster per iteration, but on small blocks its coarser residual costs SCF
# iterations: C2 converged in 11 instead of 9)
MIXED_DIIS_MIN_N = 256


# Blocks up to this size (and whose LDS footprint fits, eigh_wg_ok) are diagonalised by the
# one-workgroup-per-molecule solver of eigh.hip, which picks its thread grid by the launch's
# largest block: up to 48, 96 and 192 orbitals (EIGH_WG_CLASSES).
EIGH_WG_MAX_N = 192
EIGH_WG_LDS_DOUBLES = 20480
EIGH_WG_CLASSES = (48, 96, 192)
NUM_CU = 256  # compute units of an MI355X: the blocks of one workgroup each that run at once


def eigh_wg_lds(norb, nvec):
    """LDS doubles of the workgroup eigensolver for a launch whose largest block has norb orbitals
    and nvec vectors: the norb x nvec eigenvectors, 3 norb (diagonal, off-diagonal, eigenvalues),
    three buffers of the variant's 48 / 96 / 192 grid rows, 128 of scratch (eigh.hip lds_doubles)."""
    n = np.asarray(norb, dtype=np.int64)
    o = np.asarray(nvec, dtype=np.int64)
    slots = np.where(n <= 48, 48, np.where(n <= 96, 96, 192))
    return n * o + 3 * n + 3 * slots + 128


def eigh_wg_ok(norb, nocc):
    """Whether the workgroup eigensolver takes blocks of norb orbitals / nocc occupied orbitals:
    n <= 192 and its LDS footprint (eigh_wg_lds) fits 160 KiB (pyseqm_eigh_density_lds_ok)."""
    n = np.asarray(norb, dtype=np.int64)
    o = np.asarray(nocc, dtype=np.int64)
    return (n >= 1) & (n <= EIGH_WG_MAX_N) & (o <= n) & (eigh_wg_lds(n, o) <= EIGH_WG_LDS_DOUBLES)


def eigh_pairs_ok(norb):
    """Whether pyseqm_eigh_vectors takes every eigenpair of blocks of norb orbitals."""
    n = np.asarray(norb, dtype=np.int64)
    return (n >= 1) & (n <= EIGH_WG_MAX_N)


def size_groups(norb, ratio=0.7, min_group=32, floor=EIGH_MIN_N):
    """Partition molecules (by position) into groups of similar orbital counts: sorted by size,
    a group takes molecules down to `ratio` of its largest; groups smaller than `min_group` join
    the next larger one; sizes below `floor` count as `floor` (they are padded to it).  Returns a
    list of index arrays.  ratio 0.7 was the fastest on 1024 alkanes of 14-182 orbitals (3 groups,
    374 ms per FP64 SCF against 394 at 0.8 / 5 groups, 392 at 0.6 / 2 groups, 496 with one group):
    each batched solve costs a fixed chain of small kernels, which outweighs some padding."""
    norb = np.maximum(np.asarray(norb), floor)
    order = np.argsort(-norb, kind="stable")
    groups, start = [], 0
    while start < len(order):
        top = norb[order[start]]
        end = start
        while end < len(order) and norb[order[end]] >= ratio * top:
            end += 1
        if groups and len(groups[-1]) < min_group:
            groups[-1] = np.concatenate([groups[-1], order[start:end]])
        else:
            groups.append(order[start:end])
        start = end
    if len(groups) > 1 and len(groups[-1]) < min_group:
        groups[-2] = np.concatenate([groups[-2], groups[-1]])
        groups.pop()
    return groups


class SCFEngine:
    """Pair integrals, Fock builds, density steps and the SCF loop for one packed batch."""

    def __init__(self, species, coordinates, method, device="cuda", charges=None, batch=None, param_dir=None):
        self.device = nat.require_device(device)
        nat.lib()
        self.method = method
        self.b = batch if batch is not None else PackedBatch(species, method, self.device, charges)
        b = self.b
        dev = self.device
        f64 = dict(dtype=torch.float64, device=dev)
        tab = param_table(method, param_dir)
        self.default_params = True  # atom_par holds the parameter file's values
        par = np.zeros((b.natoms, nat.NPAR))
        par[:, :len(COLUMNS)] = tab[b.Z]
        # isolated-atom energies and atomic heats of formation (geometry independent), initial diagonal density
        Z = b.Z
        eiso = (tab[Z, 0] * np.take(USSC, Z) + tab[Z, 1] * np.take(UPPC, Z) + tab[Z, 6] * np.take(GSSC, Z)
                + tab[Z, 8] * np.take(GPPC, Z) + tab[Z, 7] * np.take(GSPC, Z) + tab[Z, 9] * np.take(GP2C, Z)
                + tab[Z, 10] * np.take(HSPC, Z))
        self.eiso_atom = eiso
        # diag_index is molecule-major in orbital order, the same order as the atoms
        guess = np.repeat(np.where(Z > 1, np.take(TORE, Z) / 4.0, 1.0), np.where(Z > 1, 4, 1))
        up = nat.upload(dev, par=par, eiso=np.bincount(b.atom_mol, eiso, minlength=b.nmol),
                        eheat=np.bincount(b.atom_mol, np.take(EHEAT, Z) / ev_kcalpmol, minlength=b.nmol),
                        diag=b.diag_index()[0].astype(np.int64), guess=guess,
                        orb_off=(np.cumsum(b.norb) - b.norb).astype(np.int64))
        self.atom_par, self.eiso, self.eheat = up["par"], up["eiso"], up["eheat"]
        self._diag, self._guess, self.orb_off = up["diag"], up["guess"], up["orb_off"]
        self.stream = nat.stream_ptr(dev)
        nat.call("pyseqm_atom_setup", b.L, nat.ptr(self.atom_par), self.stream)
        nt = b.ntiles
        self.w_xx = torch.empty(max(b.w_size[0], 1), **f64)
        self.w_xh = torch.empty(max(b.w_size[1], 1), **f64)
        self.w_hh = torch.empty(max(b.w_size[2], 1), **f64)
        self.H = torch.empty(max(b.total, 1), **f64)
        self.part = torch.empty(max(nt, 1) * 160, **f64)
        self.tile_v = torch.empty(max(nt, 1), **f64)
        self.atom_v = torch.empty(max(b.natoms, 1), **f64)
        self.enuc = torch.zeros(b.nmol, **f64)
        self.red = torch.zeros(max(b.nmol, 1) * nat.MAX_RED_BLOCKS * 16, **f64)  # reduction scratch
        self.eelec = torch.zeros(b.nmol, **f64)
        self._atoms = None
        self.coords = None
        self.trace = None  # set to a list to collect per-iteration (dE, diis, dm, dm_max) metrics
        self.diis_log = None  # set to a list to collect (cF, slot, B matrices, coefficients, resets, errors)
        self.eigh_log = collections.deque(maxlen=256)  # (blocks, largest, solver) of the recent eigensolves
        # vectors the workgroup eigensolver lost to Gram-Schmidt (stays 0 unless its vectors degenerate)
        self.eigh_fail = torch.zeros(1, dtype=torch.int32, device=dev)
        if coordinates is not None:
            self.set_coordinates(coordinates)

    # per-atom parameters the sp methods zero or derive (Molecule.py:101-113, basics.py:791-811): a
    # value passed for them does not change the reference's result either
    DERIVED_PARAMS = ("beta", "zeta_d", "s_orb_exp_tail", "p_orb_exp_tail", "d_orb_exp_tail", "U_dd", "F0SD",
                      "G2SD", "rho_core")

    def set_parameters(self, params):
        """Override per-atom MOPAC parameters ({name: (natoms,) tensor} in the batch's atom order, the
        dict Pack_Parameters returns with learned values merged in, basics.py:406-448, 781-789) and
        re-derive the multipoles, isolated-atom energies and, if coordinates are set, the integrals.
        Names the reference ignores for MNDO/AM1/PM3 are ignored; a per-pair ``Kbeta`` scaling of the
        resonance integrals (hcore.py:166-171) is not on this path and raises."""
        b = self.b
        kb = params.get("Kbeta", None)
        if torch.is_tensor(kb):
            raise NotImplementedError("per-pair Kbeta resonance scaling is not supported by the device engine")
        values = {}
        for name, v in params.items():
            if name not in COLUMNS or v is None:
                continue
            v = torch.as_tensor(v, dtype=torch.float64, device=self.device).detach().reshape(-1)
            if v.numel() != b.natoms:
                raise ValueError(f"parameter {name!r}: {v.numel()} values for {b.natoms} atoms")
            values[COLUMNS.index(name)] = v
        if len(values) == len(COLUMNS):
            self.atom_par[:, :len(COLUMNS)] = torch.stack([values[c] for c in range(len(COLUMNS))], dim=1)
        else:
            for c, v in values.items():
                self.atom_par[:, c] = v
        self.default_params = False
        nat.call("pyseqm_atom_setup", b.L, nat.ptr(self.atom_par), self.stream)
        ap = self.atom_par
        eiso = sum(ap[:, c] * coef for c, coef in self._eiso_coef())
        self.eiso_atom = eiso.cpu().numpy()
        self.eiso = torch.zeros(b.nmol, dtype=torch.float64, device=self.device).index_add_(
            0, self.atom_mol(), eiso)
        if self.coords is not None:
            self.set_coordinates(self.coords)

    def _atom_data(self):
        """Per-atom constants on the device, uploaded on first use: molecule and Eiso coefficients."""
        if self._atoms is None:
            Z = self.b.Z
            coef = [(c, np.take(t, Z).astype(np.float64)) for c, t in
                    ((0, USSC), (1, UPPC), (6, GSSC), (8, GPPC), (7, GSPC), (9, GP2C), (10, HSPC))]
            up = nat.upload(self.device, mol=self.b.atom_mol.astype(np.int64), coef=np.stack([t for _, t in coef]))
            self._atoms = up["mol"], [(c, up["coef"][k]) for k, (c, _) in enumerate(coef)]
        return self._atoms

    def atom_mol(self):
        """Molecule of each atom (int64, device)."""
        return self._atom_data()[0]

    def _eiso_coef(self):
        """(parameter column, its coefficient per atom) of the isolated-atom energy (energy.py:8-23)."""
        return self._atom_data()[1]

    # ------------------------------------------------------------- integrals
    def set_coordinates(self, coordinates, enuc_pair=False):
        """coordinates: (nmol, molsize, 3) Angstrom in the reference's padded layout, or (natoms, 3)."""
        b = self.b
        c = torch.as_tensor(coordinates, dtype=torch.float64, device=self.device)
        if c.dim() == 3:
            c = c.reshape(-1, 3)[b.d["real_flat"]]
        self.coords = c.contiguous()
        self.enuc_pair = torch.zeros(max(b.npairs, 1), dtype=torch.float64, device=self.device) if enuc_pair \
            else None
        nat.call("pyseqm_pair_integrals", b.L, nat.METHODS[self.method], nat.ptr(self.coords),
                 nat.ptr(self.atom_par), nat.ptr(self.w_xx), nat.ptr(self.w_xh), nat.ptr(self.w_hh),
                 nat.ptr(self.H), nat.ptr(self.part), nat.ptr(self.tile_v), nat.ptr(self.enuc),
                 nat.ptr(self.enuc_pair), nat.ptr(b.pair_ref_device()) if enuc_pair else None, self.stream)

    # ------------------------------------------------------------------ fock
    def fock(self, P, F, active=None, eelec=None):
        b = self.b
        out = self.eelec if eelec is None else eelec
        nat.call("pyseqm_fock", b.L, nat.ptr(self.atom_par), nat.ptr(self.w_xx), nat.ptr(self.w_xh),
                 nat.ptr(self.w_hh), nat.ptr(P), nat.ptr(self.H), nat.ptr(F), nat.ptr(self.part),
                 nat.ptr(self.tile_v), nat.ptr(self.atom_v), nat.ptr(out), nat.ptr(active), self.stream)
        return out

    def initial_density(self):
        """Diagonal guess (scf_loop.py:2066-2081): heavy atoms tore/4 on s and p, H 1.0."""
        P = torch.zeros(max(self.b.total, 1), dtype=torch.float64, device=self.device)
        P[self._diag] = self._guess
        return P

    # ---------------------------------------------------------- density step
    def density_eigh(self, F, idx, nact, Pout, want_evecs=False):
        """FP64 density step by diagonalisation of the active Fock blocks -> Pout (diag.py:110-241).

        Blocks of up to EIGH_WG_MAX_N orbitals go to the one-workgroup-per-molecule solver
        (pyseqm_eigh_density: Householder with the block in registers, multisection, twisted
        factorisations, cluster Gram-Schmidt, no padding) in one launch, those whose occupied vectors do not
        fit its LDS (28 to 32 waters; _eigh_wg_split) in one of their own.  Larger blocks, and calls
        that want the eigenvectors themselves, take the batched library eigensolver on Gershgorin-padded
        stacks, again per size group (the reference pads every molecule to the batch's largest, which for
        an uneven batch multiplies the O(n^3) work)."""
        b = self.b
        if not want_evecs:
            lds, large, rest = self._eigh_wg_split(np.asarray(self._idx_host))
            if len(lds):
                # one launch, largest blocks first: the long solves start at once and the short
                # ones fill the CUs behind them (C2's density step: 5.2 ms against 8.4 ms for
                # launches per size group, each of which waits for its own largest block)
                self._eigh_wg_run(F, *self._eigh_wg_order(lds), Pout)
            if len(large):
                self._eigh_wg_run(F, *self._eigh_wg_order(large), Pout, large=True)
            if len(rest) == 0:
                return None
            groups = size_groups(b.norb[rest])
            saved = self._idx_host
            for sel in groups:
                sub = torch.as_tensor(rest[sel].astype(np.int32), device=self.device)
                self._idx_host = rest[sel]
                self.density_eigh(F, sub, len(sel), Pout, want_evecs=True)
            self._idx_host = saved
            return None
        nmax = int(b.norb[self._idx_host].max())
        if nact >= EIGH_MIN_N_BATCH:
            nmax = max(nmax, EIGH_MIN_N)
        Fp = torch.empty(nact, nmax, nmax, dtype=torch.float64, device=self.device)
        nat.call("pyseqm_pad_for_eigh", b.L, nat.ptr(F), nat.ptr(idx), nact, nmax, nat.ptr(Fp), nat.ptr(self.red),
                 nat.red_blocks(nmax), self.stream)
        self.eigh_log.append((nact, nmax, "library"))
        e, V = torch.linalg.eigh(Fp)
        V = V.contiguous()
        nat.call("pyseqm_density_from_evecs", b.L, nat.ptr(V), nmax, nat.ptr(idx), nact, nat.ptr(Pout),
                 self.stream)
        if want_evecs:
            return e, V, nmax
        return None

    def _eigh_wg_split(self, ids):
        """Molecules `ids` by the density step that takes them: the workgroup eigensolver with its vectors in LDS, with
        its vectors in memory, the library's.  A launch asks for the LDS of its largest block and its
        highest occupation, which may be two molecules' (30 carbons, 182 / 91, and 27 waters, 162 / 108):
        blocks that fit alone but not beside the largest one go to the vectors in memory."""
        norb, nocc = self.b.norb[ids], self.b.nocc[ids]
        fits = eigh_wg_ok(norb, nocc)
        if fits.any():
            fits &= eigh_wg_ok(norb[fits].max(), nocc)
        large = ~fits & eigh_pairs_ok(norb)
        return ids[fits], ids[large], ids[~fits & ~large]

    def _eigh_wg_order(self, ids):
        """(device index list, count, largest block, most occupied orbitals) of the molecules `ids`, largest first."""
        b = self.b
        ids = ids[np.argsort(-b.norb[ids], kind="stable")]
        idx = torch.as_tensor(ids.astype(np.int32), device=self.device)
        return idx, len(ids), int(b.norb[ids[0]]), int(b.nocc[ids].max())

    def _eigh_wg_list(self, ids):
        """_eigh_wg_order of the molecules `ids` if one launch of the workgroup eigensolver takes them, else None."""
        return self._eigh_wg_order(ids) if eigh_wg_ok(self.b.norb[ids].max(), self.b.nocc[ids].max()) else None

    def _eigh_wg(self, F, ids, Pout):
        """One launch of the workgroup eigensolver on the molecules `ids` (host int array)."""
        self._eigh_wg_run(F, *self._eigh_wg_order(ids), Pout)

    def _eigh_wg_run(self, F, idx, count, nmax, nocc_max, Pout, large=False):
        ws = torch.empty((5 if large else 4) * count * nmax * nmax, dtype=torch.float64, device=self.device)
        if large:
            nat.call("pyseqm_eigh_density_large", self.b.L, nat.ptr(idx), count, nmax, nat.ptr(F), nat.ptr(Pout),
                     nat.ptr(ws), nat.ptr(ws[4 * count * nmax * nmax:]), nat.ptr(self.eigh_fail), self.stream)
        else:
            nat.call("pyseqm_eigh_density", self.b.L, nat.ptr(idx), count, nmax, nocc_max, nat.ptr(F), nat.ptr(Pout),
                     nat.ptr(ws), nat.ptr(self.eigh_fail), self.stream)
        self.eigh_log.append((count, nmax, "workgroup"))

    def _sp2_workspace(self):
        ws = getattr(self, "_sp2ws", None)
        if ws is None:
            from .sp2 import SP2Workspace
            ws = self._sp2ws = SP2Workspace(self)
        return ws

    def density(self, F, idx, nact, Pout, fixed_iters=None):
        if self.density_kind == "eigh":
            self.density_eigh(F, idx, nact, Pout)
        else:
            from . import sp2
            sp2.density_sp2(self, F, idx, nact, Pout, fixed_iters=fixed_iters)

    # ------------------------------------------------------------------- SCF
    def _active(self, notconv_host):
        idx = np.nonzero(notconv_host)[0]
        self._idx_host = idx
        return torch.as_tensor(idx.astype(np.int32), device=self.device), len(idx)

    def scf(self, eps=1e-8, converger=(2,), density="eigh", sp2_eps=1e-4, P=None, max_iter=MAX_ITER, diis_tol=None):
        """scf_loop (scf_loop.py:2034-2394) with mixers [0] linear, [1] adaptive, [2] Pulay DIIS.
        `diis_tol` overrides the max|FP - PF| convergence test (default below)."""
        b = self.b
        dev = self.device
        self.density_kind = density
        self.sp2_eps = sp2_eps
        # max|FP - PF| test: 50 eps as the reference (scf_loop.py:52); the bf16x3 SP2 density has a
        # commutator floor of ~1e-3 (its energy error stays ~1e-8 eV/atom), so it is tested at 1e-2
        self.diis_tol = 50.0 * eps if density == "eigh" else max(50.0 * eps, SP2_DIIS_TOL)
        if diis_tol is not None:
            self.diis_tol = float(diis_tol)
        f64 = dict(dtype=torch.float64, device=dev)
        P = self.initial_density() if P is None else P.clone()
        self._metrics = torch.zeros(b.nmol, 4, **f64)
        F = torch.empty_like(P)
        Pnew = torch.empty_like(P)
        e_old = torch.empty(b.nmol, **f64)
        e_new = torch.empty(b.nmol, **f64)
        self.fock(P, F, eelec=e_old)
        notconv = torch.ones(b.nmol, dtype=torch.uint8, device=dev)
        nc_host = np.ones(b.nmol, dtype=bool)
        kind = converger[0]
        it = 0
        if kind == 2:
            res = self._pulay(P, F, Pnew, e_old, e_new, notconv, eps, max_iter)
        elif kind in (0, 1):
            res = self._simple(kind, converger, P, F, Pnew, torch.zeros_like(P), e_old, e_new, notconv, eps, max_iter)
        else:
            raise ValueError("scf_converger must be [0, alpha], [1] or [2]")
        P, it, nc_host = res
        if density == "eigh":
            # the workgroup eigensolver counts eigenvectors it could not normalise (lost to their
            # cluster's span); one read per SCF
            lost = int(self.eigh_fail.item())
            if lost:
                self.eigh_fail.zero_()
                warnings.warn(f"FP64 eigensolver: {lost} eigenvector(s) lost to a cluster's span during this SCF; "
                              "the densities of the molecules involved may be inaccurate")
        out = SCFResult()
        out.P = P
        out.iterations = it
        out.notconverged = nc_host
        return out

    def _simple(self, kind, converger, P, F, Pnew, Pold, e_old, e_new, notconv, eps, max_iter):
        b = self.b
        nc_host = np.ones(b.nmol, dtype=bool)
        it = 0
        if kind == 1:
            dev = self.device
            old2 = torch.zeros(max(int(b.norb.sum()), 1), dtype=torch.float64, device=dev)  # diag of P two steps back
            orb_off = torch.as_tensor(np.concatenate([[0], np.cumsum(b.norb)[:-1]]).astype(np.int64), device=dev)
            fac = torch.zeros(b.nmol, dtype=torch.float64, device=dev)
            mask = torch.zeros(1, dtype=torch.int32, device=dev)
        krange = range(0, max_iter + 1) if kind == 0 else range(1, max_iter + 1)
        for k in krange:
            idx, nact = self._active(nc_host)
            if nact == 0:
                break
            it += 1
            nmax = int(b.norb[self._idx_host].max())
            self.density(F, idx, nact, Pnew)
            if kind == 0:
                nat.call("pyseqm_mix", b.L, nat.ptr(idx), nact, nmax, float(converger[1]), nat.ptr(P),
                         nat.ptr(Pnew), nat.ptr(Pold), self.stream)
            else:
                nat.call("pyseqm_adaptive_mix", b.L, nat.ptr(idx), nact, nmax, int(k), nat.ptr(P), nat.ptr(Pnew),
                         nat.ptr(Pold), nat.ptr(old2), nat.ptr(orb_off), nat.ptr(fac), nat.ptr(mask), self.stream)
            self.fock(P, F, active=notconv, eelec=e_new)  # notconv marks the active molecules
            nat.call("pyseqm_scf_check", b.L, nat.ptr(idx), nact, nat.ptr(P), nat.ptr(Pold), nat.ptr(e_new),
                     nat.ptr(e_old), None, float(eps), 0.0, nat.ptr(notconv), None, nat.ptr(self.red),
                     nat.red_blocks(nmax), self.stream)
            nc_host = notconv.cpu().numpy().astype(bool)
        return P, it, nc_host

    def _pulay(self, P, F, Pnew, e_old, e_new, notconv, eps, max_iter):
        """scf_forward2 (scf_loop.py:639-1132): Pulay DIIS on FP - PF with a 10-deep history,
        batch-global history counter and reset on ill-conditioning (cond > 1e7)."""
        b = self.b
        dev = self.device
        total = max(b.total, 1)
        f64 = dict(dtype=torch.float64, device=dev)
        # every element that is read is written first: a history of cF entries reads those only, and
        # pyseqm_pulay_pre starts EMAT at cF = 1
        Fring = torch.empty(NFOCK, total, **f64)
        Cring = torch.empty(NFOCK, total, **f64)
        X = torch.empty(total, **f64)
        diis_err = torch.empty(b.nmol, **f64)
        EMAT = torch.empty(b.nmol, NFOCK + 1, NFOCK + 1, **f64)
        coef = torch.empty(b.nmol, NFOCK, **f64)
        reset_flags = torch.empty(b.nmol, dtype=torch.uint8, device=dev)
        # notconv and reset flags of the last iteration: the device writes them here, pyseqm_pulay_post waits
        host = torch.empty(2, b.nmol, dtype=torch.uint8, pin_memory=True)
        status = host.numpy()
        ptrs = {k: nat.ptr(t) for k, t in dict(
            F=F, P=P, X=X, Fring=Fring, Cring=Cring, EMAT=EMAT, coef=coef, reset=reset_flags, diis=diis_err,
            red=self.red, Pnew=Pnew, par=self.atom_par, xx=self.w_xx, xh=self.w_xh, hh=self.w_hh, H=self.H,
            part=self.part, tile_v=self.tile_v, atom_v=self.atom_v, e_new=e_new, e_old=e_old, notconv=notconv,
            metrics=self._metrics, host=host).items()}
        nc_host = np.ones(b.nmol, dtype=bool)
        counter, cF = -1, 0
        it = 0
        idx = None
        for k in range(max_iter + 1):
            if idx is None:  # the active molecules changed
                idx, nact = self._active(nc_host)
                if nact == 0:
                    break
                active = self._idx_host
                nmax = int(b.norb[active].max())
                nb = nat.red_blocks(nmax)
                solver = self._eigh_wg_list(active) if self.density_kind == "eigh" else None
            it += 1
            cF = min(cF + 1, NFOCK)
            counter = (counter + 1) % NFOCK
            mixed = self.density_kind == "sp2" and nmax > MIXED_DIIS_MIN_N
            if mixed:
                # bf16x3 commutator on the upper triangle (the ring is read there only), from FP32
                # copies of F and P in the SP2 X buffers, which are free until the density step
                ws = self._sp2_workspace()
                nat.call("pyseqm_diis_commutator_bf16x3", b.L, nat.ptr(idx), nact, nmax, nat.ptr(F), nat.ptr(P),
                         nat.ptr(ws.xoff), nat.ptr(ws.xld), nat.ptr(ws.Xa), nat.ptr(ws.Xb), nat.ptr(Cring[counter]),
                         nat.ptr(diis_err), nat.ptr(self.red), nat.MAX_RED_BLOCKS * 16, self.stream)
            # the coefficients from cF = 2 on: the reference's eigh reads only the lower triangle (stale upper
            # entries included), the kernel mirrors it, normalises by B[slot][slot] and solves by FP64 Jacobi
            nat.call("pyseqm_pulay_pre", b.L, nat.ptr(idx), nact, nmax, ptrs["F"], ptrs["P"], ptrs["X"],
                     ptrs["Fring"], ptrs["Cring"], total, counter, cF, NFOCK, ptrs["EMAT"], ptrs["coef"],
                     ptrs["reset"], ptrs["diis"], ptrs["red"], nb, 0 if mixed else 1, self.stream)
            if cF >= 2 and self.diis_log is not None:
                self.diis_log.append((cF, counter, EMAT.cpu().numpy().copy(), coef.cpu().numpy().copy(),
                                      np.where(nc_host, reset_flags.cpu().numpy(), 0).astype(np.uint8),
                                      diis_err.cpu().numpy().copy()))
            if solver is not None:
                self._eigh_wg_run(F, *solver, Pnew)
            else:
                self.density(F, idx, nact, Pnew)
            nat.call("pyseqm_pulay_post", b.L, nat.ptr(idx), nact, 0.5 if cF < 2 else 0.0, ptrs["P"], ptrs["Pnew"],
                     ptrs["par"], ptrs["xx"], ptrs["xh"], ptrs["hh"], ptrs["H"], ptrs["F"], ptrs["part"],
                     ptrs["tile_v"], ptrs["atom_v"], ptrs["e_new"], ptrs["e_old"], ptrs["diis"], float(eps),
                     self.diis_tol, ptrs["notconv"], ptrs["metrics"], ptrs["red"], nb, ptrs["reset"], ptrs["host"],
                     self.stream)
            if self.trace is not None:
                self.trace.append(self._metrics.cpu().numpy().copy())
            reset = cF >= 2 and bool(status[1][active].any())
            still = status[0][active]
            if not still.all():
                nc_host[active] = still.astype(bool)
                idx = None
            if reset:
                counter, cF = -1, 0
        return P, it, nc_host

    # -------------------------------------------------------------- results
    def energies(self, P):
        """Final F = fock(P), Eelec, Enuc, Etot, Eiso, Hf per molecule (basics.py:862-892, 1220-1239)."""
        F = torch.empty_like(P)
        eelec = torch.zeros(self.b.nmol, dtype=torch.float64, device=self.device)
        self.fock(P, F, eelec=eelec)
        etot = eelec + self.enuc
        hf = etot - self.eiso + self.eheat
        return dict(F=F, Eelec=eelec, Enuc=self.enuc.clone(), Etot=etot, Eiso=self.eiso.clone(), Hf=hf)

    def forces(self, P, h=1.0e-3):
        """Forces (natoms, 3) in eV/Angstrom at fixed density P (Hellmann-Feynman, the reference's
        autograd force with scf_backward = 0, basics.py:1315-1336).  The pair gradients are closed-form:
        `h` (a step length once) has to be positive and has no other effect."""
        b = self.b
        out = torch.zeros(max(b.natoms, 1), 3, dtype=torch.float64, device=self.device)
        nat.call("pyseqm_pair_forces", b.L, nat.METHODS[self.method], nat.ptr(self.coords), nat.ptr(self.atom_par),
                 nat.ptr(P), float(h), nat.ptr(self.part), nat.ptr(out), self.stream)
        return out[:b.natoms]

    def param_grad(self, P, hrel=1.0e-4, atom_par=None, coords=None):
        """Derivatives of the energy at fixed density P with respect to every atom's 24 input
        parameters (COLUMNS order): (natoms, 2, 24), [:, 0] for Eelec and [:, 1] for the core
        repulsion Enuc.  At a converged SCF density this is the exact gradient of Etot (the energy is
        stationary in P), the one the reference's autograd returns for learned parameters with
        scf_backward = 0 (basics.py:781-789, scf_loop.py:1996-2031).  Pair and one-center terms in
        closed form; the derivatives of each atom's multipoles in its inputs are 4th-order central
        differences (step hrel * max(|value|, 0.1)).  atom_par / coords default to the engine's current ones."""
        b = self.b
        out = torch.zeros(max(b.natoms, 1), 2, 24, dtype=torch.float64, device=self.device)
        rec = torch.empty(max(int(nat.lib().pyseqm_param_grad_workspace(nat.ctypes.byref(b.L))), 1),
                          dtype=torch.float64, device=self.device)
        ap = self.atom_par if atom_par is None else atom_par.contiguous()
        xyz = self.coords if coords is None else coords.contiguous()
        nat.call("pyseqm_param_grad", b.L, nat.METHODS[self.method], nat.ptr(xyz), nat.ptr(ap),
                 nat.ptr(P), float(hrel), nat.ptr(rec), nat.ptr(self.part), nat.ptr(out), self.stream)
        return out[:b.natoms]

    def eiso_grad(self):
        """d(isolated-atom energy)/d(input parameter) per atom, (natoms, 24): the coefficients of
        U_ss, U_pp, g_ss, g_sp, g_pp, g_p2, h_sp in Eiso (energy.py:8-23)."""
        b = self.b
        g = torch.zeros(b.natoms, 24, dtype=torch.float64, device=self.device)
        for c, coef in self._eiso_coef():
            g[:, c] = coef
        return g

    def eigenpairs(self, F, orb_off, evals, Q, eig_ws, fail):
        """Every eigenpair of every block of F: Q in the packed layout (column j = eigenvector j,
        ascending eigenvalues) and evals[orb_off[m] + j].  Blocks of up to EIGH_WG_MAX_N orbitals take
        pyseqm_eigh_vectors, in one launch for those whose vectors fit its LDS (at most 139 orbitals) and
        one for the others, or in one for all where every block has a CU of its own; larger ones the
        batched library eigensolver on Gershgorin-padded stacks per size group, scattered into the same
        layout.  eig_ws: scratch that a launch may overwrite whole, of 4 nmol n^2 doubles for the n of the
        workgroup blocks, or None to allocate each launch's here (as where it is smaller); fail counts
        vectors the workgroup solver lost (read by the caller)."""
        b = self.b
        norb = np.asarray(b.norb)
        wg = eigh_pairs_ok(norb)
        in_lds = eigh_wg_ok(norb, norb)
        if int(wg.sum()) <= NUM_CU and not in_lds[wg].all():
            # the small blocks run beside the large ones (us, two launches -> one: 128 alkanes of 14-182 orbitals
            # 1020 -> 615, 255 blocks of 14 and one of 140 503 -> 439, of 192 747 -> 680, 250 of 139 and one of
            # 140 892 -> 481, 200 of 50 and 56 of 182 745 -> 632, 250 of 96 and 6 of 140 686 -> 464)
            in_lds = np.zeros_like(in_lds)
        for ids in (np.nonzero(wg & ~in_lds)[0], np.nonzero(in_lds)[0]):
            if len(ids) == 0:
                continue
            ids = ids[np.argsort(-norb[ids], kind="stable")]  # long solves first, as in density_eigh
            top = int(norb[ids[0]])
            need = 4 * len(ids) * top ** 2
            ws = eig_ws if eig_ws is not None and eig_ws.numel() >= need else torch.empty(
                need, dtype=torch.float64, device=self.device)
            idx = torch.as_tensor(ids.astype(np.int32), device=self.device)
            nat.call("pyseqm_eigh_vectors", b.L, nat.ptr(idx), len(ids), top, nat.ptr(F), nat.ptr(orb_off),
                     nat.ptr(evals), nat.ptr(Q), nat.ptr(ws), nat.ptr(fail), self.stream)
        rest = np.nonzero(~wg)[0]
        if len(rest) == 0:
            return
        off_h = np.concatenate([[0], np.cumsum(norb)[:-1]]).astype(np.int64)
        for sel in size_groups(norb[rest]):
            g = rest[sel]
            nmax = int(norb[g].max())
            idx = torch.as_tensor(g.astype(np.int32), device=self.device)
            Fp = torch.empty(len(g), nmax, nmax, dtype=torch.float64, device=self.device)
            nat.call("pyseqm_pad_for_eigh", b.L, nat.ptr(F), nat.ptr(idx), len(g), nmax, nat.ptr(Fp),
                     nat.ptr(self.red), nat.red_blocks(nmax), self.stream)
            e0, V = torch.linalg.eigh(Fp)  # padded eigenvalues lie above each block's spectrum
            for k, m in enumerate(g):
                n = int(norb[m])
                o = int(b.mol_mat_off[m])
                Q[o:o + n * n].view(n, n).copy_(V[k, :n, :n])
                evals[int(off_h[m]):int(off_h[m]) + n].copy_(e0[k, :n])

    def eig(self, F):
        """Orbital energies in the reference layout e (nmol, 4*molsize), zero padded, and the packed
        eigenvectors (nmol, nmax, nmax), sym_eig_trunc(eig_only=True) (diag.py:110-241).  Batches of
        blocks of up to EIGH_WG_MAX_N orbitals take the workgroup eigensolver (128 alkanes of 14-182
        orbitals: 1.2 ms, 6.5 by the library's batched solver; energies and squared vector elements are as
        exact as the library's); those with a larger block, or where the
        workgroup solver lost a vector or met a value that is not finite, the library's."""
        b = self.b
        self._idx_host = np.arange(b.nmol)
        nmax = b.nmax
        f64 = dict(dtype=torch.float64, device=self.device)
        if eigh_pairs_ok(b.norb).all():
            fail = torch.zeros(1, dtype=torch.int32, device=self.device)
            evals = torch.empty(int(b.norb.sum()), **f64)
            Q = torch.empty(max(b.total, 1), **f64)
            self.eigenpairs(F, self.orb_off, evals, Q, None, fail)
            e = torch.empty(b.nmol, 4 * b.molsize, **f64)
            V = torch.empty(b.nmol, nmax, nmax, **f64)
            nat.call("pyseqm_evec_view", b.L, b.molsize, nmax, nat.ptr(self.orb_off), nat.ptr(evals),
                     nat.ptr(Q), nat.ptr(e), nat.ptr(V), nat.ptr(fail), self.stream)
            if int(fail.item()) == 0:
                return e, V
        idx = torch.arange(b.nmol, dtype=torch.int32, device=self.device)
        Fp = torch.empty(b.nmol, nmax, nmax, **f64)
        nat.call("pyseqm_pad_for_eigh", b.L, nat.ptr(F), nat.ptr(idx), b.nmol, nmax, nat.ptr(Fp),
                 nat.ptr(self.red), nat.red_blocks(nmax), self.stream)
        e0, V = torch.linalg.eigh(Fp)
        e = torch.zeros(b.nmol, 4 * b.molsize, **f64)
        mask = torch.arange(nmax, device=self.device)[None, :] < torch.as_tensor(b.norb, device=self.device)[:, None]
        e[:, :nmax] = torch.where(mask, e0, torch.zeros_like(e0))
        return e, V

    # ------------------------------------------------- reference-order views
    def w_reference(self):
        """Two-center integrals as the reference's dense (npairs, 10, 10) array (hcore.py:9-179)."""
        b = self.b
        w = torch.empty(b.npairs, 10, 10, dtype=torch.float64, device=self.device)
        nat.call("pyseqm_w_reference", b.L, nat.ptr(b.pair_base_device()), nat.ptr(self.w_xx), nat.ptr(self.w_xh),
                 nat.ptr(self.w_hh), nat.ptr(w), nat.stream_ptr(self.device))
        return w

    def orbital_charges(self, V):
        """Per-orbital charge on each atom (nmol, 4 molsize, molsize) from the eigenvectors (nmol, n, n)
        (scf_loop.py:2376-2387)."""
        b = self.b
        out = torch.empty(b.nmol, 4 * b.molsize, b.molsize, dtype=torch.float64, device=self.device)
        nat.call("pyseqm_orbital_charges", b.L, b.molsize, nat.ptr(V), V.stride(0), V.stride(1), V.stride(2),
                 nat.ptr(out), nat.stream_ptr(self.device))
        return out
