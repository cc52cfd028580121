"""GPU: calls whose vectors pass through pinned memory (up to 64 KB each way) against
the same work copied, and the q-space memory that is kept between calls, with batches
growing and shrinking and from several threads at once.  The kernels are the same on
both paths: equal results, bit for bit."""
import threading

import numpy as np
import pytest

from tests.systems import random_block_system, random_perturbation

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [45, 88, 89, 90])   # 4 chains, 1, 1 and none fit
def test_averages(n):
    from tdscha_amd.engine import Engine
    s = random_block_system(n, 60, 2, [1] * n, seed=n)
    eng = Engine(s["X"], s["Y"], s["w"], s["rho"], s["T"], s["syms"], s["blocks"], s["sbi"])
    R, Y = (np.stack(a) for a in zip(*(random_perturbation(n, seed=k) for k in range(8))))
    f, d = eng.perturb_averages_batched(R, Y)
    for k in range(8):
        fk, dk = eng.perturb_averages(R[k], Y[k])
        assert np.array_equal(fk, f[k]) and np.array_equal(dk, d[k])
    f3, d3 = eng.perturb_averages_batched(R[:3], Y[:3])
    assert np.array_equal(f3, f[:3]) and np.array_equal(d3, d[:3])
    eng.close()


def test_apply_L():
    import types

    from tdscha_amd.lanczos import Lanczos
    for n in (45, 89, 91):
        s = random_block_system(n, 50, 1, [1] * n, seed=n)
        lanc = Lanczos(types.SimpleNamespace(T=s["T"], w=s["w"], pols=np.eye(n), m=np.ones(n),
                                             N=50, rho=s["rho"], X=s["X"], Y=s["Y"]))
        lanc.init(use_symmetries=False)
        x = np.random.default_rng(n).normal(size=(8, n + n * (n + 1)))
        y = lanc.apply_L_batch(x)
        for k in range(8):
            assert np.array_equal(lanc.apply_L_batch(x[k])[0], y[k])
        lanc.close()


def test_q_space_memory():
    from tdscha_amd import qspace as QS
    from tdscha_amd.qlanczos import QSpaceEngine
    rng = np.random.default_rng(0)
    L, N, nb = 2, 50, 6
    nq = L ** 3
    X, Y = (rng.normal(size=(nq, N, nb)) + 1j * rng.normal(size=(nq, N, nb)) for _ in range(2))
    valid = np.ones((nb, nq), bool)
    valid[:3, 0] = False
    eng = QSpaceEngine(X, Y, rng.uniform(2e-4, 2e-3, (nb, nq)), valid, np.ones(N), 300.0)
    work = []
    for C in (1, 8, 3, 20, 2):
        iq = [int(q) for q in rng.integers(0, nq, C)]
        pms = [QS.pair_map(L, q)[0] for q in iq]
        psis = [(lambda n: rng.normal(size=n) + 1j * rng.normal(size=n))(eng.psi_size(pm))
                for pm in pms]
        work.append((iq, pms, psis, eng.apply_L(iq, pms, psis)))
    for iq, pms, psis, ref in work[::-1]:
        assert all(np.array_equal(a, b) for a, b in zip(eng.apply_L(iq, pms, psis), ref))
    bad = []

    def run(k):
        for _ in range(10):
            iq, pms, psis, ref = work[k]
            if not all(np.array_equal(a, b) for a, b in zip(eng.apply_L(iq, pms, psis), ref)):
                bad.append(k)

    threads = [threading.Thread(target=run, args=(k,)) for k in range(len(work))]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    eng.close()
    assert not bad


def test_network_forward():
    from tdscha_amd.terminator import Network, forward_many, init_params
    for dims in ([80, 128, 10], [300, 300, 300]):
        nets = [Network(dims[0], dims[1], 1, dims[2], max_batch=m,
                        params=init_params(dims, np.random.default_rng(m))) for m in (250, 7)]
        x = np.random.default_rng(1).normal(size=(263, dims[0])).astype(np.float32)
        y = forward_many(nets, x)
        for k, net in enumerate(nets):
            one = np.concatenate([net.forward(x[i:i + 1]) for i in range(len(x))])
            assert np.array_equal(net.forward(x), one) and np.array_equal(y[k], one)
            net.close()
