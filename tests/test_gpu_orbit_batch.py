"""GPU: a chain's form, and its result bit for bit, does not depend on its batch.
Perturbations with a small orbit (IR vectors, Raman tensors of rank 6: more pairs than
one pass takes) and without one, together and alone.

In FP16x2 the kernels fold one row-dot into the matrix product, whose rounding (2^-22 a
term) differs between the places of the three chains that they take at once: there the
form is the same and the results agree to 1e-6, the accuracy of the split averages."""
import numpy as np
import pytest

from tests.test_gpu_orbit_runs import System

pytestmark = pytest.mark.gpu


def tensors(p, kinds, seed=2):
    """Symmetric matrices sum_ij a_ij v_i v_j^T of the x, y, z vectors, a symmetric:
    "A" the unit matrix, "E" diagonal and traceless, "T" off the diagonal; the images of
    a sum of them span 1, 2 and 3 directions each."""
    rng = np.random.default_rng(seed)
    V = np.array([(p.ens.ir_vector(e) / np.sqrt(p.ens.m)) @ p.ens.pols for e in np.eye(3)])
    out = []
    for kind in kinds:
        d, t = rng.normal(size=3), rng.normal(size=(3, 3))
        a = np.zeros((3, 3))
        if "A" in kind:
            a += np.eye(3)
        if "E" in kind:
            a += np.diag(d - d.mean())
        if "T" in kind:
            a += np.triu(t, 1) + np.triu(t, 1).T
        Y = V.T @ a @ V
        out.append(Y / np.linalg.norm(Y))
    return np.array(out)


def batch(p):
    """R, Y of eight chains: IR, none, Raman, IR with Raman, none, Raman (3 times)."""
    rng = np.random.default_rng(4)
    ir, z = p.ir(), np.zeros((p.n, p.n))
    G = rng.normal(size=(2, p.n, p.n)) / p.n
    Y = tensors(p, ["AET"] * 4)
    R = np.array([ir[0], rng.normal(size=p.n), 0 * ir[0], ir[1], ir[2], 0 * ir[0], 0 * ir[0],
                  0 * ir[0]])
    return R, np.array([z, G[0] + G[0].T, Y[0], z, G[1] + G[1].T, Y[1], Y[2], Y[3]]), 6


def same(x, y, prec):
    return np.array_equal(x, y) if prec != "fp16x2" else (
        np.linalg.norm(x - y) <= 1e-6 * np.linalg.norm(y))


@pytest.mark.parametrize("prec, N, form", [("fp64", 3000, "images"), ("fp64", 3001, "operators"),
                                           ("fp16x2", 7000, "images"), ("bf16x2", 7000, "images")])
def test_batch_equals_single_calls(prec, N, form):
    p = System(N=N, reference=False, form=form)
    lanc = p.sides[0]
    lanc.precision, eng = prec, lanc.engine
    R, Y, orbit = batch(p)
    f, d = eng.perturb_averages_batched(R, Y, 1, prec)
    assert eng.orbit_chains() == orbit
    for c in range(8):
        fc, dc = eng.perturb_averages_batched(R[c:c + 1], Y[c:c + 1], 1, prec)
        assert eng.orbit_chains() == (c not in (1, 4))
        assert same(fc[0], f[c], prec) and same(dc[0], d[c], prec)
    x = p.pack(R, Y, Y[::-1])       # another relation than Y1's in a run
    y = lanc.apply_L_batch(x)
    runs = p.pack(R, Y, 0.5 * Y)
    a, _ = lanc.run_FT_batched(np.concatenate([runs, runs[:3]]), 4)
    assert eng.orbit_chains() == orbit + 2
    for c in range(8):
        assert same(lanc.apply_L_batch(x[c:c + 1])[0], y[c], prec)
        single, _ = lanc.run_FT_batched(runs[c:c + 1], 4, use_graph=False)
        for other in [a[c]] + ([a[8 + c]] if c < 3 else []):
            assert all(same(u, v, prec) for u, v in zip(single[0], other))
    p.close()


def test_five_tensors_keep_the_form():
    p = System(reference=False)
    Y = tensors(p, ["AET"] * 5)
    p.sides[0].engine.perturb_averages_batched(np.zeros((5, p.n)), Y, 1)
    assert p.sides[0].engine.orbit_chains() == 5
    p.close()
