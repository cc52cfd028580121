"""GPU: the d2v blocks and the final sums of the q-space application in slices.

Grids of 1, 8 and 27 q-points with 6 or 3 bands give every slab length (16, 8 and 4
configurations) in both forms, matrix instructions (6 bands) and a thread per item (3
bands), 64 q-points the longest item lists;
configuration counts below one slab, at its edges and with several chunks; batches
with fewer items than a work-group and more.  Against the direct form of d2v (one
pair and chunk per work-group) on the same engine: FP64 sums of the same terms in
another order, 1e-12 norm-wise as the other FP64 tests; a chain alone equals itself in
a batch exactly."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("L, nb, N, C", [(1, 6, 3, 1), (1, 3, 40, 70), (2, 6, 15, 3), (2, 6, 16, 8),
                                         (2, 6, 17, 40), (2, 6, 3001, 9), (3, 6, 4, 5),
                                         (3, 6, 130, 30), (3, 3, 31, 11), (4, 6, 33, 12)])
def test_slices(L, nb, N, C):
    from tdscha_amd import qspace as QS
    from tdscha_amd.qlanczos import QSpaceEngine
    rng = np.random.default_rng(N)
    nq = L ** 3
    X, Y = (rng.normal(size=(nq, N, nb)) + 1j * rng.normal(size=(nq, N, nb)) for _ in range(2))
    w = rng.uniform(2e-4, 2e-3, size=(nb, nq))
    valid = np.ones((nb, nq), bool)
    valid[:3, 0] = False
    eng = QSpaceEngine(X, Y, w, valid, rng.uniform(0.5, 1.5, N), 300.0)
    iq = [int(q) for q in rng.integers(0, nq, C)]
    pms = [QS.pair_map(L, q)[0] for q in iq]
    psis = [(lambda n: rng.normal(size=n) + 1j * rng.normal(size=n))(eng.psi_size(pm))
            for pm in pms]
    out = eng.apply_L(iq, pms, psis)
    one = eng.apply_L(iq[-1:], pms[-1:], psis[-1:])
    eng.set_d2v_form(0)
    ref = eng.apply_L(iq, pms, psis)
    eng.close()
    for o, r in zip(out, ref):
        assert np.linalg.norm(o - r) <= 1e-12 * np.linalg.norm(r)
    if N <= 64:   # a single chunk whatever the batch
        assert np.array_equal(one[0], out[-1])
