"""The trainer's loss over a batch whose blocks take hundreds of tiles each."""
import numpy as np
import pytest

from dmx import abi
from dmx import learned

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("target", [0.9, 0.7])
def test_loss_of_a_large_batch_keeps_its_digits(target):
    """2^20 rows (256 tiles a block), zero parameters, so that every output is
    0 and all terms 0.5 target^2 / n are the same number: a running float32 sum
    of them is off by 1.3e-6 and more, always to one side.  A term has one
    rounding (the square; the half and the division by 2^20 are exact) and the
    loss another, 2^-24 each."""
    n = 1 << 20
    print(f"[gpu] loss of {n} rows, target {target}", flush=True)
    m = abi.Mlp(n)
    m.set_params(np.zeros(learned.NPARAM, np.float32))
    T = np.full((n, 8), target, np.float32)
    loss, _ = m.loss_grad(np.zeros((n, 40), np.float32), T)
    want = 4.0 * float(T[0, 0]) ** 2
    assert abs(loss / want - 1.0) <= 2.0 ** -22
    m.close()
