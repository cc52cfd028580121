"""GPU: the orbit form (perturbations whose rotated images span a few directions)
against the general form, on rock salt with its point group.

The general form is reached through a context without symmetries whose
configurations are the images S_j x_i themselves (fewer than four symmetries: no
orbit form), and through the range entry of the same context.  Tolerances: the
relation of the images is accepted to 1e-12 of the largest image and its weakest
direction is at least 1e-3 of it, so averages agree to 1e-9; a chain adds one such
term per step, and the general form loses the symmetry sector by about a factor 5
per step from rounding (5^8 x 1e-15): 1e-8 on the coefficients of 8 steps."""
import copy

import numpy as np
import pytest

from tests.test_rotation_form import dense_syms

pytestmark = pytest.mark.gpu

AXES = ((1.0, 0.0, 0.0), (0.0, 1.0, 0.0), (0.3, -0.5, 0.8))


def rel(a, b):
    return np.linalg.norm(a - b) / np.linalg.norm(b)


class Pair:
    """The same system with its symmetries and with its images as configurations."""

    def __init__(self, L, N, gamma, form="images", wigner=True, drop=0):
        from tdscha_amd.lanczos import Lanczos
        from tdscha_amd.rocksalt import Ensemble, RockSalt
        ens = Ensemble(RockSalt(L=L), 300.0, N, seed=L)
        ms = ens.symmetries(True, gamma_only=gamma)
        if drop:
            ms = copy.copy(ms)
            ms.symmetries = [s[:-drop] for s in ms.symmetries]
        self.ms, self.n, self.N = ms, len(ens.w), N
        self.n_syms = ms.symmetries[0].shape[0]
        S = dense_syms(ms.symmetries, ms.degenerate_space, self.n)
        img = copy.copy(ens)
        img.X = np.concatenate([ens.X @ s.T for s in S])
        img.Y = np.concatenate([ens.Y @ s.T for s in S])
        img.rho, img.N = np.ones(len(img.X)), len(img.X)
        one = copy.copy(ms)
        one.symmetries = [np.ones((1, 1, 1))] * self.n
        one.degenerate_space = [np.array([i], dtype=np.int32) for i in range(self.n)]
        one.sym_block_id = np.arange(self.n, dtype=np.int32)
        self.sides = []
        for e, m, f in ((ens, ms, form), (img, one, "images")):
            lanc = Lanczos(ens, use_wigner=wigner)
            lanc.X, lanc.Y, lanc.rho, lanc.N = e.X, e.Y, e.rho, e.N
            lanc.N_eff = float(np.sum(e.rho))
            lanc.gamma_only = gamma
            lanc.symmetry_form = f
            lanc.init(symmetries=m)
            self.sides.append(lanc)
        self.ens = ens

    def starts(self):
        out = []
        for pv in AXES:
            self.sides[0].prepare_perturbation(self.ens.ir_vector(pv), masses_exp=-1)
            out.append(self.sides[0].psi / np.linalg.norm(self.sides[0].psi))
        return np.array(out)

    def close(self):
        for lanc in self.sides:
            lanc.close()


def sector_perturbations(ms, r0, nc):
    """R1, Y1 of nc members of the sector of the IR vector r0: a random vector and a
    random symmetric matrix projected by the point group, rotated by its members."""
    rng = np.random.default_rng(7)
    n = len(r0)
    S = dense_syms(ms.symmetries, ms.degenerate_space, n)
    A = rng.normal(size=(n, n))
    chi = S @ r0 @ r0 / (r0 @ r0)
    Y = np.einsum("j,jab,bc,jdc->ad", chi, S, A + A.T, S, optimize=True)
    R = np.einsum("j,jab,b->a", chi, S, rng.normal(size=n), optimize=True)
    k = rng.integers(0, len(S), nc)
    return (np.array([S[j].T @ R for j in k]),
            np.array([S[j].T @ Y @ S[j] for j in k]))


CASES = [(3, 1900, True, "images"), (3, 1901, True, "operators"), (2, 2710, False, "images")]


@pytest.mark.parametrize("L, N, gamma, form", CASES)
def test_averages(L, N, gamma, form):
    p = Pair(L, N, gamma, form)
    a, b = (s.engine for s in p.sides)
    for nc, d4, prec in ((3, 1, 0), (3, 0, 0), (8, 1, 1), (8, 1, 2)):
        R, Y = sector_perturbations(p.ms, p.starts()[0][:p.n], nc)
        f, d = a.perturb_averages_batched(R, Y, d4, prec)
        if prec == 0:
            fo, do = b.perturb_averages_batched(R, Y, d4, 0)
            assert rel(f, fo) < 1e-9 and rel(d, do) < 1e-9
            assert np.abs(d - np.transpose(d, (0, 2, 1))).max() == 0.0
        else:   # too little work in the split precisions: the general form
            fr, dr = a.perturb_averages_range(R, Y, 1, p.N * p.n_syms, d4, prec)
            assert np.array_equal(f, fr) and np.array_equal(d, dr)
        # one member without symmetry: the general form, as over the whole range
        R[-1] = np.random.default_rng(1).normal(size=p.n)
        f, d = a.perturb_averages_batched(R, Y, d4, prec)
        fr, dr = a.perturb_averages_range(R, Y, 1, p.N * p.n_syms, d4, prec)
        assert np.array_equal(f, fr) and np.array_equal(d, dr)
    p.close()


@pytest.mark.parametrize("rotate", [False, True])
@pytest.mark.parametrize("prec, tol", [(0, 1e-9), (1, 1e-6), (2, 1e-5)])
def test_averages_of_many_images(prec, tol, rotate):
    """Enough images that the split precisions take the orbit form (7 pairs and more:
    two groups): against the FP64 average over the whole range of the images, within
    the accuracy of the split products (2^-22 and 2^-17 per term, as the other split
    tests), and no further from it than the general form in the same precision."""
    from tdscha_amd.engine import Engine
    from tdscha_amd.rocksalt import Ensemble, RockSalt
    ens = Ensemble(RockSalt(L=3), 300.0, 11000, seed=5)
    ms = ens.symmetries(True, gamma_only=True)
    v = (ens.ir_vector() / np.sqrt(ens.m)) @ ens.pols
    R, Y = sector_perturbations(ms, v, 8)
    eng = Engine(ens.X, ens.Y, ens.w, np.ones(ens.N), 300.0, ms.symmetries, ms.degenerate_space,
                 ms.sym_block_id, rotate=rotate)
    f, d = eng.perturb_averages_batched(R, Y, 1, prec)
    M = ens.N * ms.symmetries[0].shape[0]
    fo, do = eng.perturb_averages_range(R, Y, 1, M, 1, 0)
    fg, dg = eng.perturb_averages_range(R, Y, 1, M, 1, prec)
    eng.close()
    assert rel(f, fo) < tol and rel(d, do) < tol
    if prec:
        assert rel(f, fo) + rel(d, do) < rel(fg, fo) + rel(dg, do)


@pytest.mark.parametrize("wigner, transpose", [(True, False), (False, False), (False, True)])
@pytest.mark.parametrize("L, N, gamma, form", CASES)
def test_apply_L(L, N, gamma, form, wigner, transpose):
    p = Pair(L, N, gamma, form, wigner)
    x = p.starts()
    y = p.sides[1].apply_L_batch(x, transpose)
    assert rel(p.sides[0].apply_L_batch(x, transpose), y) < 1e-9
    y2 = p.sides[1].apply_L_batch(y, transpose)
    assert rel(p.sides[0].apply_L_batch(y, transpose), y2) < 1e-9
    p.close()


@pytest.mark.parametrize("drop", [0, 1])     # 1: not a group, the general form
@pytest.mark.parametrize("L, N, gamma, form", CASES)
def test_chains(L, N, gamma, form, drop):
    p = Pair(L, N, gamma, form, drop=drop)
    x, caps = p.starts(), [3, 8, 5]
    ref, _ = p.sides[1].run_FT_batched(x, 8, caps=caps)
    runs = [p.sides[0].run_FT_batched(x, 8, caps=caps, use_graph=g)[0]
            for g in (False, "step", "run")]
    for g in runs:
        for (a, b), (ao, bo), (a0, b0), cap in zip(g, ref, runs[0], caps):
            assert len(a) == len(ao) == cap
            assert np.abs(a / ao - 1).max() < 1e-8 and np.abs(b / bo - 1).max() < 1e-8
            assert np.array_equal(a, a0) and np.array_equal(b, b0)
    p.close()


def test_long_chains_stay_in_their_sector():
    """The three IR chains of a cubic crystal are equal by symmetry.  In FP64 their
    converged spectra agree to the rounding that the recurrence amplifies (4e-8 to 1e-7
    in the general form); rounding that leaves the sector unchecked shows as 3e-6.
    Tolerance: ten times the general form's, 1e-6."""
    from tdscha_amd.lanczos import Lanczos, continued_fraction
    from tdscha_amd.rocksalt import RY_TO_CM, Ensemble, RockSalt
    ens = Ensemble(RockSalt(L=4), 300.0, 20000, seed=0)
    lanc = Lanczos(ens)
    lanc.use_wigner, lanc.gamma_only = True, True
    lanc.init(use_symmetries=True)
    psis = []
    for pv in np.eye(3):
        lanc.prepare_perturbation(ens.ir_vector(pv), masses_exp=-1)
        psis.append(lanc.psi.copy())
    w = np.linspace(0.0, 600.0, 2000) / RY_TO_CM
    S = [-np.imag(continued_fraction(a, b, None, w, True, use_terminator=False,
                                     smearing=5.0 / RY_TO_CM))
         for a, b in lanc.run_FT_batched(np.array(psis), 200, reorth=True)[0]]
    lanc.close()
    for s in S[1:]:
        assert np.abs(s - S[0]).max() < 1e-6 * np.abs(S[0]).max()
