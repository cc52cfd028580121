"""GPU: network passes with every layer in one kernel, at the edges of their panels
(128 of each index), widths (256) and depth (8 layers), of the rows of a work-group and
of the grid slices of the spectral loss, and one size past each on the separate
kernels, against the CPU oracle.  Tolerances as in the other network tests: FP32
kernels against FP64, 1e-4 of the largest output, 2e-3 of a layer's largest gradient."""
import numpy as np
import pytest

from oracle import mlp_oracle as MO

pytestmark = pytest.mark.gpu


def relerr(x, ref):
    return float(np.max(np.abs(x - ref)) / np.max(np.abs(ref)))


def make(dims, hidden, seed, max_batch):
    from tdscha_amd.terminator import Network, init_params
    p = (init_params(dims, np.random.default_rng(seed)) * 2.0).astype(np.float32)
    return p, Network(dims[0], dims[1] if hidden else 1, hidden, dims[-1], params=p,
                      max_batch=max_batch)


@pytest.mark.parametrize("n_in, width, hidden, n_out, B", [
    (1, 1, 0, 1, 1), (5, 3, 0, 7, 6), (127, 128, 1, 129, 5), (128, 129, 2, 10, 4),
    (129, 127, 1, 1, 7), (256, 256, 7, 256, 9), (200, 255, 3, 130, 33), (257, 64, 1, 10, 8),
    (16, 16, 8, 10, 8), (40, 32, 2, 10, 4099)])
def test_layers(n_in, width, hidden, n_out, B):
    dims = [n_in] + [width] * hidden + [n_out]
    p, net = make(dims, hidden, n_in, B)
    rng = np.random.default_rng(B)
    x = rng.normal(size=(B, n_in)).astype(np.float32)
    t = rng.normal(size=(B, n_out)).astype(np.float32)
    y = net.forward(x)
    yo, _, _ = MO.forward(p.astype(np.float64), dims, x.astype(np.float64))
    assert relerr(y, yo) < 1e-4
    loss, g = net.loss_grad(0, x, target=t)
    lo, go = MO.mse_loss_grad(p.astype(np.float64), dims, x.astype(np.float64),
                              t.astype(np.float64), np.ones(n_out))
    assert loss == pytest.approx(lo, rel=1e-4)
    off = 0
    for l in range(len(dims) - 1):
        n = dims[l + 1] * dims[l] + dims[l + 1]
        assert relerr(g[off:off + n], go[off:off + n]) < 2e-3, l
        off += n
    net.close()


@pytest.mark.parametrize("K, B, n_w", [(1, 1, 1), (7, 3, 255), (8, 2, 256), (9, 5, 257),
                                       (20, 3, 2049), (17, 700, 800)])
def test_spectral_slices(K, B, n_w):
    dims = [2 * K, 16, 10]
    p, net = make(dims, 1, K, B)
    rng = np.random.default_rng(n_w)
    a = -0.5 + 0.05 * rng.normal(size=(B, K))
    b = rng.uniform(0.08, 0.12, (B, K))
    w = np.linspace(0.1, 1.2, n_w)
    mean = np.r_[-5.0, 1.0, np.zeros(8)]
    std = np.full(10, 0.3)
    ref = rng.uniform(0.0, 1.0, (B, n_w))
    x = rng.normal(size=(B, 2 * K)).astype(np.float32)
    ch = np.concatenate([a, b, b[:, :1], np.full((B, 1), 0.1)], axis=1)
    net.set_cf_loss(K, w, 0.02, mean, std, 10.0)
    loss, g = net.loss_grad(1, x, chains=ch, ref=ref)
    lo, go = MO.cf_batch_loss_grad(p.astype(np.float64), dims, x.astype(np.float64), ch, ref, w,
                                   0.02, mean, std, 10.0, K)
    assert loss == pytest.approx(lo, rel=1e-4)
    assert relerr(g, go) < 2e-3
    net.close()
