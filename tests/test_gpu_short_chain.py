"""GPU: the recurrence of short chains in one work-group against the separate kernels.

The line between them is the number of steps asked for (entries of the whole basis),
so a run with a step cap far above its chain's cap takes the separate kernels for the
same chain.  Lengths at the edges of the register rows (1024 entries, 256 complex ones)
and one or all rows; stops by cap, by tolerance and by a start vector in a small
invariant space.  Tolerance: full reorthogonalisation keeps the coefficients of a few
steps to rounding, 1e-10 as the other chain tests."""
import numpy as np
import pytest

from tests.systems import random_block_system

pytestmark = pytest.mark.gpu


def close(x, y):
    for (a, b), (ao, bo) in zip(x, y):
        assert len(a) == len(ao) and len(b) == len(bo)
        assert np.abs(a / ao - 1).max() < 1e-10
        assert len(b) == 0 or np.abs(b / bo - 1).max() < 1e-10


@pytest.mark.parametrize("reorth", [True, False])
@pytest.mark.parametrize("n", [1, 2, 30, 31, 32, 54, 55, 77])
def test_mode_space(n, reorth):
    import types

    from tdscha_amd.lanczos import Lanczos
    s = random_block_system(n, 40, 1, [1] * n, seed=n)
    ens = types.SimpleNamespace(T=s["T"], w=s["w"], pols=np.eye(n, n), m=np.ones(n), N=40,
                                rho=s["rho"], X=s["X"] * 0.02, Y=s["Y"] * 1e-2)
    lanc = Lanczos(ens)
    lanc.init(use_symmetries=False)
    len_ = n + n * (n + 1)
    x = np.random.default_rng(n).normal(size=(3, len_))
    x[2, 1:] = 0.0
    caps = [min(6, len_ - 1), 1, min(4, len_ - 1)]
    long = min(1536, 300001 // len_ + 1)
    runs = [lanc.run_FT_batched(x, m, caps=caps, reorth=reorth, use_graph=g)[0]
            for m, g in ((8, False), (8, "step"), (long, "step"))]
    close(runs[0], runs[1])
    close(runs[0], runs[2])
    lanc.close()


@pytest.mark.parametrize("L, nb", [(1, 3), (1, 6), (2, 6), (3, 3), (3, 6), (4, 6)])
def test_q_space(L, nb):
    from tdscha_amd import qspace as QS
    from tdscha_amd.qlanczos import QSpaceEngine
    rng = np.random.default_rng(L)
    nq, N = L ** 3, 40
    X, Y = (rng.normal(size=(nq, N, nb)) + 1j * rng.normal(size=(nq, N, nb)) for _ in range(2))
    w = rng.uniform(2e-4, 2e-3, size=(nb, nq))
    valid = np.ones((nb, nq), bool)
    valid[:3, 0] = nq == 1
    eng = QSpaceEngine(X, 1e-8 * Y, w, valid, np.ones(N), 300.0)
    iq = [int(q) for q in rng.integers(0, nq, 3)]
    pms = [QS.pair_map(L, q)[0] for q in iq]
    psis = []
    for pm in pms:
        p = np.zeros(eng.psi_size(pm), complex)
        p[:nb] = rng.normal(size=nb) + 1j * rng.normal(size=nb)
        psis.append(p)
    ld = max(len(p) for p in psis)
    caps = [5, 1, 4]
    runs = [[(a, b) for a, b, c in eng.lanczos(iq, pms, psis, m, caps=caps, use_graph=g)[0]]
            for m, g in ((6, False), (6, True), (min(1024, 150001 // ld + 1), False))]
    close(runs[0], runs[1])
    close(runs[0], runs[2])
    eng.close()
