"""The float64 HLLD solvers with shared reciprocals (hlld1d_fast, hlld2d_fast)
and their fallback outside the operand range: bit for bit the oracle, sign of
zero included, where fields, velocities or pressures are zero, of order one,
tiny (the products of two fields vanish), denormal, or huge, cell by cell in
turn, so that lanes of one wave take both forms."""
import numpy as np
import pytest

import oracle as O
from dmx import abi
from dmx import problems as P

pytestmark = pytest.mark.gpu

# (field scale, velocity scale, pressure scale, only every other column)
CASES = [(0.0, 1.0, 1.0, False), (1e-70, 1.0, 1.0, False), (1e-120, 1.0, 1.0, True), (1e-205, 1.0, 1.0, False),
         (1e-212, 0.0, 1.0, True), (1e-300, 1e-230, 1.0, False), (1e-315, 1e-318, 1.0, True), (1.0, 1e-200, 1.0, True),
         (1.0, 0.0, 1.0, False), (1.0, 1.0, 1e-25, False), (1e-9, 1e-9, 1e-18, True), (1e16, 1e16, 1e32, False),
         (1e15, 1e15, 1e30, True), (-1.0, 1e-160, 1.0, False)]


@pytest.mark.parametrize("case", range(len(CASES)))
def test_fp64_hlld_out_of_range_matches_oracle_bitwise(case):
    bs, vs, ps, alternate = CASES[case]
    pb = P.random_smooth(19, 10, 7, seed=60 + case, mach=0.5, beta=2.0)
    p, u = pb.params, pb.uin.copy()
    print(f"[gpu] HLLD range: field {bs}, velocity {vs}, pressure {ps}, alternate {alternate}", flush=True)
    pres = np.zeros(u.shape[1:])
    pres[3:-3, 3:-3, 3:-3] = P.pressure(p, u)
    j = np.arange(p.ny + 6)
    on = (j // 2 % 2 == 0 if alternate else j >= 0)[None, :, None]
    vel = [np.where(on, vs, 1.0) * u[1 + c] / u[0] for c in range(3)]
    b = [np.where(on, bs, 1.0) * u[5 + c] for c in range(3)]
    inner = (slice(3, -3),) * 3
    v = P.assemble(p, u[0][inner], *(c[inner] for c in vel), (ps * pres)[inner], *(c[inner] for c in b))
    o, d = O.Oracle(p, v), abi.Domain(p, v)
    t = 0.0
    for _ in range(2):
        t_o, dts_o = o.advance(1, t)
        t_g, dts_g = d.advance(1, t)
        t = t_o
        assert np.array_equal(dts_o, dts_g) and t_o == t_g
        got, want = P.interior(d.download()), P.interior(o.store())
        bad = got.view(np.int64) != want.view(np.int64)
        bad &= ~(np.isnan(got) & np.isnan(want))
        assert not bad.any(), (int(bad.sum()), got[bad][:4], want[bad][:4])
    d.close()
