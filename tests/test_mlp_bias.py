"""Bias gradients of the network at the edges of the summation's tiles (128
rows, 64 columns) against the NumPy reference."""
import numpy as np
import pytest

import mlp_ref


@pytest.mark.gpu
@pytest.mark.parametrize("n", [1, 127, 128, 129, 1000])
@pytest.mark.parametrize("width", [5, 64, 65, 200])
def test_bias_gradient_sizes(n, width):
    from sccm_amd.surrogate import MLP
    rng = np.random.default_rng(n + width)
    sizes = [14, width, 3]
    net = MLP(sizes, seed=3)
    X = rng.normal(size=(n, 14)).astype(np.float32)
    Y = rng.normal(size=(n, 3)).astype(np.float32)
    net.set_data(X, Y)
    loss, g = net.loss_grad(np.arange(n))
    lr, gr = mlp_ref.loss_grad(net.get_params().astype(np.float64), sizes, X, Y)
    assert abs(loss - lr) <= 1e-5 * abs(lr)
    assert np.abs(g - gr).max() <= 1e-4 * np.abs(gr).max()  # the tolerance of the gradient test
    net.close()
