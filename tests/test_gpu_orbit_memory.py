"""GPU: the memory of the orbit form.  Its partial sums are the context's, whatever their
K split; its workspaces give way to an allocation that finds no room, and come back."""
import numpy as np
import pytest

from tests.device_memory import free_bytes
from tests.test_gpu_orbit_batch import tensors
from tests.test_gpu_orbit_runs import System

pytestmark = pytest.mark.gpu


def test_partial_sums_of_the_context():
    p = System(reference=False)
    eng = p.sides[0].engine
    Y = tensors(p, ["AET"] * 5)
    z = np.zeros((5, p.n))
    f, d = eng.perturb_averages_batched(z, Y, 1)
    for ks in (8, 16, 256):
        eng.set_ksplit(ks)
        fk, dk = eng.perturb_averages_batched(z, Y, 1)
        assert eng.orbit_chains() == 5
        assert np.array_equal(f, fk) and np.array_equal(d, dk)
    p.close()


@pytest.mark.parametrize("prec, N", [("fp64", 3000), ("fp16x2", 7000)])
def test_workspaces_give_way(prec, N):
    from tdscha_amd._lib import TdschaError
    p = System(N=N, reference=False)
    lanc = p.sides[0]
    lanc.precision = prec
    x = p.pack(p.ir())
    y = lanc.apply_L_batch(x)
    free = free_bytes()
    with pytest.raises(TdschaError):     # 64 chains of 100,000 steps: a petabyte
        lanc.run_FT_batched(np.tile(x[:1], (64, 1)), 100000, use_graph=False)
    assert free_bytes() - free > 20 << 20
    again = lanc.apply_L_batch(x)
    assert lanc.engine.orbit_chains() == 3 and np.array_equal(again, y)
    p.close()
