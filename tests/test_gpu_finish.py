"""GPU: sums, symmetrisation and output of calls of one column tile in one launch, at
the edges of its 8 x 8 blocks and 64-mode rows of f, in every form of L, against the
oracle.  Tolerance: FP64 sums in another order, the 1e-12 norm-wise bound of the other
L tests.  More than 256 partials take the separate kernels."""
import types

import numpy as np
import pytest

from tests.systems import random_block_system

pytestmark = pytest.mark.gpu


def rel(a, b):
    return np.linalg.norm(a - b) / np.linalg.norm(b)


@pytest.mark.parametrize("n", [1, 7, 8, 9, 45, 64, 65, 120, 127, 128])
def test_forms(n):
    from oracle import lanczos_oracle as O
    from tdscha_amd.lanczos import Lanczos
    s = random_block_system(n, 70, 1, [1] * n, seed=n)
    X, Y = s["X"] * 0.02, s["Y"] * 1e-2
    ens = types.SimpleNamespace(T=s["T"], w=s["w"], pols=np.eye(n, n), m=np.ones(n), N=70,
                                rho=s["rho"], X=X, Y=Y)
    vecs = np.random.default_rng(n).normal(size=(3, n + n * (n + 1)))
    for wigner in (True, False):
        lanc = Lanczos(ens)
        lanc.use_wigner = wigner
        lanc.init(use_symmetries=False)
        orc = O.OracleSystem(X, Y, s["w"], s["rho"], s["T"], np.eye(n)[None], use_wigner=wigner)
        for transpose in (False, True):
            if wigner and transpose:
                continue
            ref = [orc.apply_full_L(v, transpose=transpose) for v in vecs]
            got = lanc.apply_L_batch(vecs, transpose=transpose)
            for g, r in zip(got, ref):
                assert rel(g, r) < 1e-12
            lanc.reverse_L, lanc.shift_value = True, 0.25
            for v, r in zip(vecs, ref):
                assert rel(lanc.apply_full_L(v.copy(), transpose=transpose), 0.25 * v - r) < 1e-12
            lanc.reverse_L, lanc.shift_value = False, 0.0
        lanc.close()


@pytest.mark.parametrize("ks", [8, 16, 24, 56, 128, 248, 256, 512])
def test_partials(ks):
    """Every number of partials, also where a slice of the sums is ragged or empty."""
    from oracle import c_oracle as CO
    from tdscha_amd.engine import Engine
    from tests.systems import random_perturbation
    n, N = 21, 300
    s = random_block_system(n, N, 1, [1] * n, seed=3)
    eng = Engine(s["X"], s["Y"], s["w"], s["rho"], s["T"], s["syms"], s["blocks"], s["sbi"])
    eng.set_ksplit(ks)
    R1, Y1 = random_perturbation(n, seed=ks)
    f, d = eng.perturb_averages(R1, Y1, 1)
    eng.close()
    fo, do = CO.oracle_perturb_averages(s["X"], s["Y"], s["w"], s["rho"], R1, Y1, s["T"], 1,
                                        s["syms"], s["blocks"], s["sbi"])
    assert rel(f, fo) <= 1e-12 and rel(d, do) <= 1e-12
