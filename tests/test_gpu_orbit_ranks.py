"""GPU: the orbit form at every rank of a Raman tensor, with weights other than one, in
the image and the operator form, and its chains in the split precisions.

Reference: the images as configurations (the general form).  FP64 averages to 1e-12,
as the other FP64 tests; coefficients of 8 FP64 steps to 1e-8 (rounding of 1e-15 grows
by about 5 per step).  Split products are good to about 1e-6 (FP16x2) and 1e-5 (BF16x2)
of the averages (as the split tests ask): ten times that for 4 steps."""
import numpy as np
import pytest

from tests.test_gpu_orbit_batch import tensors
from tests.test_gpu_orbit_runs import System

pytestmark = pytest.mark.gpu

RANKS = {"A": 1, "E": 2, "T": 3, "AE": 3, "AT": 4, "ET": 5, "AET": 6}


def rel(a, b):
    return np.linalg.norm(a - b) / np.linalg.norm(b)


@pytest.mark.parametrize("form", ["images", "operators"])
def test_ranks_and_weights(form):
    p = System(weights=np.random.default_rng(6).uniform(0.2, 2.0, 3001), N=3001, form=form)
    a, b = (s.engine for s in p.sides)
    Y = tensors(p, list(RANKS))
    z = np.zeros((len(Y), p.n))
    for kind, y in zip(RANKS, Y):
        S = p.S
        W = np.array([(s.T @ y @ s).ravel() for s in S])
        assert np.linalg.matrix_rank(W, tol=1e-9) == RANKS[kind]
    for d4 in (0, 1):
        f, d = a.perturb_averages_batched(z, Y, d4)
        assert a.orbit_chains() == len(Y)
        fo, do = b.perturb_averages_batched(z, Y, d4)
        for k in range(len(Y)):
            assert rel(f[k], fo[k]) < 1e-12
            assert rel(d[k], do[k]) < 1e-12 if d4 else not d[k].any()
    p.check(p.pack(z, Y, 0.3 * Y), len(Y))
    p.close()


def test_384_operations():
    p = System(N=3000, full=True, trans=False)
    a, b = (s.engine for s in p.sides)
    Y = tensors(p, list(RANKS))
    z = np.zeros((len(Y), p.n))
    d = a.perturb_averages_batched(z, Y, 1)[1]     # (f of a tensor is zero by symmetry)
    assert a.orbit_chains() == len(Y)
    do = b.perturb_averages_batched(z, Y, 1)[1]
    for k in range(len(Y)):
        assert rel(d[k], do[k]) < 1e-12
    Y, R = p.sector(p.ir()[0], 5, 3)
    f, d = a.perturb_averages_batched(R, Y, 1)
    assert a.orbit_chains() == 3
    fo, do = b.perturb_averages_batched(R, Y, 1)
    assert rel(f, fo) < 1e-12 and rel(d, do) < 1e-12
    p.check(p.pack(p.ir()), 3)
    p.close()


@pytest.mark.parametrize("prec, tol", [("fp16x2", 1e-5), ("bf16x2", 1e-4)])
def test_split_chains(prec, tol):
    p = System(N=7000)
    Y = tensors(p, ["AET", "T"])
    x = np.concatenate([p.pack(p.ir()), p.pack(np.zeros((2, p.n)), Y, 0.3 * Y)])
    ref, _ = p.sides[1].run_FT_batched(x, 4)
    out, _ = p.sides[0].run_FT_batched(x, 4, precision=prec)
    assert p.sides[0].engine.orbit_chains() == 5
    for (a, b), (ao, bo) in zip(out, ref):
        assert np.abs(a / ao - 1).max() < tol and np.abs(b / bo - 1).max() < tol
    p.close()
