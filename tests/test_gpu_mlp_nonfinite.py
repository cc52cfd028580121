"""GPU: infinities and NaN in the network's rows, at widths that fill the fused kernels'
panels and that do not: as in plain FP32 products over the layer's own width."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n_in, width, n_hidden", [(3, 20, 2), (5, 128, 3), (7, 130, 3),
                                                   (12, 250, 1), (9, 300, 2)])
def test_rows_with_infinities_and_nan(n_in, width, n_hidden):
    from tdscha_amd.terminator import Network, init_params
    dims = [n_in] + [width] * n_hidden + [10]
    p = np.abs(init_params(dims, np.random.default_rng(width)))
    net = Network(n_in, width, n_hidden, 10, params=p)
    x = np.abs(np.random.default_rng(1).normal(size=(6, n_in))).astype(np.float32)
    good = net.forward(x)
    assert np.all(np.isfinite(good))
    x[1, 0] = np.inf              # positive weights: every output is infinite
    x[3] = 3e38                   # overflows in a hidden layer
    x[4, -1] = np.nan
    y = net.forward(x)
    assert np.all(np.isposinf(y[1])) and np.all(np.isposinf(y[3])) and np.all(np.isnan(y[4]))
    assert np.array_equal(y[[0, 2, 5]], good[[0, 2, 5]])
    net.close()
