"""The face/edge stage with one Riemann problem of a cell per block
(k_flux_split, taken over one plane per block on small domains) against the
kernel that solves the six problems in one thread: the same bits in both
precisions, for every solver, and on both sides of the line where it stops."""
import numpy as np
import pytest

from dmx import abi
from dmx import problems as P

pytestmark = pytest.mark.gpu

# the last is over the float64 line (6161 blocks of one plane), under float32's
CASES = [dict(n=(19, 7, 5)), dict(n=(62, 9, 11), riemann=P.HLL, riemann2d=P.LLF, slope_type=1),
         dict(n=(61, 5, 4), riemann=P.LLF, riemann2d=P.UPWIND, bdtype=(P.ZERO_GRADIENT, P.PERIODIC, P.ZERO_GRADIENT)),
         dict(n=(33, 8, 3), riemann=P.UPWIND, riemann2d=P.HLLA, slope_type=0), dict(n=(4, 400, 60))]


@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("case", range(len(CASES)))
def test_split_equals_one_thread_per_cell(case, precision):
    kw = dict(CASES[case])
    pb = P.random_smooth(*kw.pop("n"), seed=80 + case, precision=precision, **kw)
    print(f"[gpu] split face/edge stage, case {case}, precision {precision}", flush=True)
    out = []
    for kz in (1, 2):
        d = abi.Domain(pb.params, pb.uin)
        d.set_shape((0, kz), (0, 4))
        d.advance(2, 0.0)
        out.append(d.download())
        d.close()
    assert np.array_equal(out[0], out[1])
