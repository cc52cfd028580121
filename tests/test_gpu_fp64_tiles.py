"""FP64 averages at the edges of the column tiles (16 CB columns, ceil(n / 128)
tiles), of the 64-row and 8-row chunks and of the copy rings, against the C
oracle.  Tolerance: sums of up to n^2 N terms of FP64 products in another order,
the 1e-12 norm-wise bound of the other FP64 tests."""
import numpy as np
import pytest

from oracle import c_oracle as CO
from tests.systems import random_block_system, random_perturbation

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n, N", [(1, 3), (15, 1), (16, 7), (17, 64), (33, 65), (48, 130), (64, 9),
                                  (65, 200), (80, 33), (81, 127), (96, 70), (97, 128), (112, 40),
                                  (113, 77), (127, 129), (128, 63), (129, 90), (159, 201),
                                  (257, 50)])
def test_tile_edges(n, N):
    from tdscha_amd.engine import Engine
    s = random_block_system(n, N, 2, [1] * n, seed=n)
    eng = Engine(s["X"], s["Y"], s["w"], s["rho"], s["T"], s["syms"], s["blocks"], s["sbi"])
    R1, Y1 = random_perturbation(n, seed=N)
    f, d = eng.perturb_averages(R1, Y1, 1)
    fo, do = CO.oracle_perturb_averages(s["X"], s["Y"], s["w"], s["rho"], R1, Y1, s["T"], 1,
                                        s["syms"], s["blocks"], s["sbi"])
    # three chains in one launch, over a range with partial tiles at both ends
    Rs, Ys = np.stack([R1, 2 * R1, -R1]), np.stack([Y1, 0.5 * Y1, Y1])
    parts = [eng.perturb_averages_range(Rs, Ys, a, b) for a, b in
             ((1, max(1, N // 3)), (max(1, N // 3) + 1, 2 * N))]
    eng.close()
    assert np.linalg.norm(f - fo) <= 1e-12 * np.linalg.norm(fo)
    assert np.linalg.norm(d - do) <= 1e-12 * np.linalg.norm(do)
    fr, dr = (sum(p[k] for p in parts) for k in (0, 1))
    assert np.linalg.norm(fr[0] - fo) <= 1e-12 * np.linalg.norm(fo)
    assert np.linalg.norm(dr[0] - do) <= 1e-12 * np.linalg.norm(do)
    assert np.linalg.norm(fr[1] - 0.5 * fo) <= 1e-12 * np.linalg.norm(fo)
