"""The majorant's kernels at the row counts where they split their work differently: inference tiles of 16 rows,
steps of four tiles from 65536 rows on, the last one ragged; gradient rows of eight tiles and their last tile.
Compared with the CPU oracle, with the bounds of the other majorant tests: FP32 accumulation order inside the
matrix cores and rare BF16 flips of a hidden value."""
import numpy as np
import pytest

from oracle import majorant as M
from test_gpu_majorant import dev, rand_data, rand_params

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 15, 16, 17, 63, 64, 65, 65535, 65536, 65537, 70001])
def test_inference_rows(gpu, n):
    from gamedev_amd import Majorant
    print(f"[majorant] inference n={n}", flush=True)
    X, _, norm = rand_data(n, n)
    p = rand_params(n)
    m = Majorant("fiducial_3d", seed=1)
    m.set_params(p, norm)
    x = dev(X, gpu)
    y = m.infer(x).cpu().numpy()
    yo = M.predict(p, norm, X)
    rel = np.abs(y - yo)/yo
    assert np.median(rel) < 2e-5 and rel.max() < 5e-3, (np.median(rel), rel.max())
    # a row's output depends on its own inputs alone: the same bits in a block of another size
    k = min(n, 200)
    assert np.array_equal(m.infer(x[n - k:].contiguous()).cpu().numpy(), y[n - k:])


@pytest.mark.parametrize("n", [81903, 81919, 81920, 81921, 81985])
def test_inference_rows_either_kernel(gpu, n):
    """Both sides of the row count from which a wavefront takes four tiles in a loop instead of one, and the same
    bits from either kernel."""
    from gamedev_amd import Majorant
    print(f"[majorant] inference n={n}", flush=True)
    X, _, norm = rand_data(n, n)
    p = rand_params(n)
    m = Majorant("fiducial_3d", seed=1)
    m.set_params(p, norm)
    x = dev(X, gpu)
    y = m.infer(x).cpu().numpy()
    yo = M.predict(p, norm, X)
    rel = np.abs(y - yo)/yo
    assert np.median(rel) < 2e-5 and rel.max() < 5e-3, (np.median(rel), rel.max())
    for k in (17, 16384):
        assert np.array_equal(m.infer(x[n - k:].contiguous()).cpu().numpy(), y[n - k:])
    double = m.infer(x.repeat(2, 1)).cpu().numpy()
    assert np.array_equal(double[:n], y) and np.array_equal(double[n:], y)


@pytest.mark.parametrize("n", [1, 15, 16, 17, 127, 128, 129, 1025])
def test_gradient_rows(gpu, n):
    from gamedev_amd import Majorant
    print(f"[majorant] gradient n={n}", flush=True)
    X, lt, norm = rand_data(100 + n, n)
    p = rand_params(7)
    m = Majorant("fiducial_3d", seed=1)
    m.set_params(p, norm)
    g, loss = m.grad(dev(X, gpu), dev(lt, gpu))
    go, lo = M.loss_grad(p, norm, X, lt)
    assert abs(loss - lo) <= 1e-4*abs(lo) + 1e-6
    # one flip of a hidden value's last BF16 bit (2^-8) moves a sample's gradient by that share of it
    scale = np.abs(go).max()
    assert np.abs(g - go).max() <= max(2e-3, 2**-8/n)*scale + 1e-7
    assert float(np.dot(g, go)/np.linalg.norm(g)/np.linalg.norm(go)) > 0.9999


@pytest.mark.parametrize("n,batch", [(1, 1), (2, 1), (3, 2), (255, 50), (256, 64), (257, 64), (513, 100), (5000, 1000)])
def test_training_order(gpu, n, batch):
    """Two epochs of minibatches in the oracle's shuffled order, one Adam step at 1e-2 each: a sample in another
    minibatch would move parameters by a good part of the step."""
    from gamedev_amd import Majorant
    print(f"[majorant] training order n={n} batch={batch}", flush=True)
    X, lt, norm = rand_data(300 + n, n)
    p0 = rand_params(11)
    m = Majorant("fiducial_3d", seed=1)
    m.set_params(p0, norm)
    losses = m.train(dev(X, gpu), dev(lt, gpu), epochs=2, batch=batch, lr=1e-2, seed=77)
    p, _ = m.params()
    po, lo = M.train(p0, norm, X, lt, epochs=2, batch=batch, lr=1e-2, seed=77)
    # epoch losses to the rounding of a minibatch's BF16 activations; parameters except where a gradient near
    # zero changes sign under that rounding
    np.testing.assert_allclose(losses, lo, rtol=2e-3, atol=1e-6)
    assert np.quantile(np.abs(p - po), 0.9) < 2e-3


@pytest.mark.parametrize("n", [1, 2, 31, 32, 33, 16383, 16385, 200001])
def test_feature_statistics(gpu, n):
    """Column means and deviations of device rows against NumPy in FP64: sums of n rounded terms in two orders, the
    constant column exactly constant."""
    from gamedev_amd import Majorant
    X, _, _ = rand_data(500 + n, n)
    X[:, 3] = 2.5
    X[:, 5] = 1e6 + X[:, 5]
    m = Majorant("fiducial_3d", seed=1)
    mu, sd = m._column_stats(dev(X, gpu))
    x = X.astype(np.float64)
    scale = np.abs(x).max(axis=0)
    assert np.all(np.abs(mu - x.mean(axis=0)) <= n*2**-53*scale)
    assert np.all(np.abs(sd - x.std(axis=0)) <= 4*n*2**-53*scale)
    assert mu[3] == 2.5 and sd[3] == 0.0
    norm = m.fit_normalization(dev(X, gpu))
    assert norm[8 + 3] == 1.0
