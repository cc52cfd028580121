"""GPU: the scales of the split averages (Y1, the folded column of R1, B) at the edges
of the mode padding, where the folded column exists (n < 128 k) and where it does not,
with R1 and Y1 of very different size, against FP64 on the same engine.  Tolerances:
those of the split averages, 2e-5 (FP16x2) and 2e-3 (BF16x2) norm-wise."""
import numpy as np
import pytest

from tests.systems import random_block_system, random_perturbation

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n, N", [(1, 40), (127, 300), (128, 257), (129, 1000), (256, 128)])
@pytest.mark.parametrize("scale", [1.0, 1e-6, 1e6])
def test_scales(n, N, scale):
    from tdscha_amd.engine import Engine
    s = random_block_system(n, N, 1, [1] * n, seed=n)
    eng = Engine(s["X"], s["Y"], s["w"], s["rho"], s["T"], s["syms"], s["blocks"], s["sbi"])
    R1, Y1 = random_perturbation(n, seed=N)
    Rs, Ys = np.stack([R1, scale * R1]), np.stack([Y1, Y1])
    ref = eng.perturb_averages_batched(Rs, Ys, 1)
    for prec, tol in ((1, 2e-5), (2, 2e-3)):
        got = eng.perturb_averages_batched(Rs, Ys, 1, precision=prec)
        for g, r in zip(got, ref):
            for c in range(2):
                assert np.linalg.norm(g[c] - r[c]) <= tol * np.linalg.norm(r[c])
    eng.close()
