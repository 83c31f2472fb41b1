"""FARGO advection in a domain whose y boundaries are not periodic: the ghost
rows beside the wrapped rows are then no images of them, and the remap reads the
two source rows' neighbours separately.  Against the oracle bit for bit, with
shifts over several rows, so that source rows lie on both sides of the wrap."""
import numpy as np
import pytest

import oracle as O
from dmx import abi
from dmx import problems as P

pytestmark = pytest.mark.gpu

# x in [-1, 1]: both signs of the shift
CASES = [dict(n=(7, 9, 5), omega0=12.0), dict(n=(5, 65, 4), slope_type=1, omega0=8.0),
         dict(n=(12, 4, 3), slope_type=0, omega0=16.0), dict(n=(9, 33, 3), slope_type=3, omega0=10.0),
         dict(n=(6, 40, 4), iso=1, ciso=1.0, omega0=12.0)]


@pytest.mark.parametrize("x", [P.PERIODIC, P.ZERO_GRADIENT])
@pytest.mark.parametrize("case", range(len(CASES)))
def test_fargo_between_walls(case, x):
    kw = dict(CASES[case])
    pb = P.random_smooth(*kw.pop("n"), seed=500 + case, xmin=-1.0, xmax=1.0)
    p = pb.params.replace(bdtype=(x, P.ZERO_GRADIENT, P.PERIODIC), fargo=1, **kw)
    print(f"[gpu] FARGO between walls, case {case}, x boundary {x}", flush=True)
    o = O.Oracle(p, pb.uin)
    t_o, dts_o = o.advance(3)
    # the outer columns' shift in rows
    assert (1.5 * p.omega0 * p.xmax * dts_o * p.ny).max() > 1.0
    d = abi.Domain(p, pb.uin)
    t_g, dts_g = d.advance(3, 0.0)
    assert t_o == t_g and np.array_equal(dts_o, dts_g)
    inner = (slice(None, 8), slice(3, -3), slice(3, -3), slice(3, -3))
    got, want = d.download(), o.store()
    assert np.isfinite(want[inner]).all()
    assert np.array_equal(got[inner], want[inner]), float(np.abs(got - want)[inner].max())
    d.close()
