"""The surrogate's gradient where its matrix products divide unevenly: partial
tiles and partial slices of both tile sizes, one row, one hidden unit, and a
batch whose forward products take the larger tiles (260 of them, five over
the hidden units by 52 over the rows)."""
import numpy as np
import pytest

from test_gpu_surrogate import _random_net, mlp_ref

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nin,H,M", [
    (1, 1, 1), (5, 33, 129), (31, 65, 31), (3, 129, 257), (3, 260, 3300)])
def test_gradient_at_uneven_sizes(nin, H, M):
    print("[gpu-surrogate-size] %d %d %d" % (nin, H, M), flush=True)
    net, w = _random_net(nin, H, seed=nin + H)
    rng = np.random.default_rng(11)
    xmean = np.zeros(nin, dtype=np.float32)
    xstd = np.ones(nin, dtype=np.float32)
    net.set_standardization(xmean, xstd, 0.0, 1.0)
    x = rng.normal(size=(M, nin)).astype(np.float32)
    y = rng.normal(size=M)
    loss, g = net.loss_grad(x, y)
    lref, gref = mlp_ref.loss_grad(w, net.offsets, nin, H, x.astype(np.float64),
                                   y.astype(np.float32).astype(np.float64))
    # the bounds of the tested sizes; with one row a value that float rounding
    # carries over a bfloat16 tie (2^-9 of it) is not averaged over others
    few = 20 if M == 1 else 1
    assert loss == pytest.approx(lref, rel=1e-4 * few)
    scale = np.max(np.abs(gref))
    np.testing.assert_allclose(g, gref, rtol=1e-3 * few, atol=1e-3 * few * scale)
