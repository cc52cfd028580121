"""GPU: the q-space batch memory that a context keeps between calls is bounded: a batch
that needs more than 1 GiB gives it back."""
import numpy as np
import pytest

from tests.device_memory import free_bytes

pytestmark = pytest.mark.gpu


def test_kept_memory_is_bounded():
    from tdscha_amd import qspace as QS
    from tdscha_amd.qlanczos import QSpaceEngine
    rng = np.random.default_rng(0)
    L, N, nb, C = 2, 150000, 6, 256     # weights of the configurations: 1.2 GB
    nq = L ** 3
    X = rng.normal(size=(nq, N, nb)) + 1j * rng.normal(size=(nq, N, nb))
    valid = np.ones((nb, nq), bool)
    valid[:3, 0] = False
    eng = QSpaceEngine(X, X[:, ::-1], rng.uniform(2e-4, 2e-3, (nb, nq)), valid, np.ones(N), 300.0)
    iq = [int(q) for q in rng.integers(0, nq, C)]
    pms = [QS.pair_map(L, q)[0] for q in iq]
    psis = [(lambda n: rng.normal(size=n) + 1j * rng.normal(size=n))(eng.psi_size(pm))
            for pm in pms]
    small = eng.apply_L(iq[:3], pms[:3], psis[:3])
    free = free_bytes()
    out = eng.apply_L(iq, pms, psis)
    assert free - free_bytes() < 1 << 30
    again = eng.apply_L(iq[:3], pms[:3], psis[:3])
    for a, b in zip(small, again):
        assert np.array_equal(a, b)
    assert all(np.all(np.isfinite(o)) for o in out)
    eng.close()
