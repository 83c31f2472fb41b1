"""Launch shapes at the ends of the accepted domain sizes."""
import numpy as np
import pytest

from dmx import abi
from dmx import problems as P

pytestmark = pytest.mark.gpu


def test_long_thin_box_splits_within_the_grid_limit():
    """One block of columns over 12000 planes: over one plane per block the
    six problems of a cell would take 72006 blocks along z, more than a grid
    has, so one thread solves them; as created, over one plane, over two, and
    through the tuner."""
    pb = P.random_smooth(3, 3, 12000, seed=12, precision=1)
    print("[gpu] long thin box", flush=True)
    out = []
    for shape in (None, (0, 1), (0, 2)):
        d = abi.Domain(pb.params, pb.uin)
        if shape:
            d.set_shape(shape, (0, 4))
        d.advance(2, 0.0)
        out.append(d.download())
        d.close()
    assert np.array_equal(out[0], out[2]) and np.array_equal(out[1], out[2])
    d = abi.Domain(pb.params, pb.uin)
    d.tune()
    _, dts = d.advance(2, 0.0)
    assert np.isfinite(dts).all() and np.isfinite(d.download()[:8]).all()
    d.close()
