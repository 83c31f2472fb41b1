"""The trainer's fused forward and backward kernel at batch sizes around its
tiles of 16 rows and its 256 blocks (one row, a ragged last tile, several
tiles per block) against the float64 reference."""
import numpy as np
import pytest

from dmx import abi
from dmx import learned

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 15, 16, 17, 4095, 4097, 8200])
def test_forward_loss_gradient_match_reference(n):
    """To 1e-4 of the largest component, as float32 sums over 64 inputs and n rows."""
    g = np.random.Generator(np.random.PCG64(n))
    X = g.uniform(-1.0, 1.0, (n, 40)).astype(np.float32)
    T = g.normal(0.0, 0.3, (n, 8)).astype(np.float32)
    th = (learned.init_params(5) + 0.05 * g.standard_normal(learned.NPARAM)).astype(np.float32)
    print(f"[gpu] training tiles, {n} rows", flush=True)
    m = abi.Mlp(8200)
    m.set_params(th)
    y = learned.forward(th, X)
    assert np.abs(m.forward(X) - y).max() <= 1e-5 * np.abs(y).max()
    loss, grad = m.loss_grad(X, T)
    want, gwant = learned.loss_and_grad(th, X, T)
    assert abs(loss - want) <= 1e-5 * want
    assert np.abs(grad - gwant).max() <= 1e-4 * np.abs(gwant).max()
    m.close()
