"""GPU: the orbit form of the averages when R1 and Y1 differ in size.  f depends on Y1
alone, and without d4 d2v depends on R1 alone: a relation of the images counts only if
it holds for each of them to its own size.  Reference: the images as configurations
(the general form); tolerance 1e-12, as for the other FP64 averages."""
import numpy as np
import pytest

from tests.test_gpu_orbit_runs import System

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("scale", [1.0, 1e-8, 1e-16, 1e-24])
def test_parts_of_different_size(scale):
    p = System()
    a, b = (s.engine for s in p.sides)
    rng = np.random.default_rng(1)
    R = p.ir()
    Y, r = p.sector(R[0], 5, 3)
    G = rng.normal(size=(3, p.n, p.n)) / p.n
    g = rng.normal(size=(3, p.n)) / np.sqrt(p.n)
    cases = (
        (r, scale * Y, 1, 3), (scale * r, Y, 0, 3),      # both in one sector: rank 3
        (R[1] * scale, Y, 0, 3), (R[1], scale * Y, 1, 3),   # other members of it: rank 6
        (r, 0 * Y, 1, 3), (0 * r, Y, 0, 3),
        (r, scale * (G + G.transpose(0, 2, 1)), 1, 0), (scale * g, Y, 0, 0))   # none
    for R1, Y1, d4, orbit in cases:
        R1 = np.broadcast_to(R1, (3, p.n))
        f, d = a.perturb_averages_batched(R1, Y1, d4)
        assert a.orbit_chains() == orbit
        fo, do = b.perturb_averages_batched(R1, Y1, d4)
        for x, xo in ((f, fo), (d, do)):
            assert np.linalg.norm(x - xo) <= 1e-12 * np.linalg.norm(xo)
    p.close()
