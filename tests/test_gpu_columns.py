"""Kernels that cut a domain into columns of their own: the FARGO advection
(256 consecutive cells a block), the shearing ghosts (64 rows a block) and the
viscous fluxes (tiles of at most 33 x 16 columns, 2 to 8 planes), against the
oracle bit for bit at the edges of their tiles; the launch shapes of a context
as created; and a state carried through the transfers, which stage it where the
trace summary lies."""
import numpy as np
import pytest

import oracle as O
from dmx import abi
from dmx import learned
from dmx import problems as P

pytestmark = pytest.mark.gpu


def _same(pb, p, steps):
    o = O.Oracle(p, pb.uin)
    t_o, dts_o = o.advance(steps)
    d = abi.Domain(p, pb.uin)
    t_g, dts_g = d.advance(steps, 0.0)
    assert t_o == t_g and np.array_equal(dts_o, dts_g)
    inner = (slice(None, 8), slice(3, -3), slice(3, -3), slice(3, -3))
    got, want = d.download(), o.store()
    assert np.array_equal(got[inner], want[inner]), float(np.abs(got - want)[inner].max())
    d.close()


# rows shorter and longer than the box's shift, one block and a ragged second
# one, ny on both sides of 64, every slope type the remap knows
SHEAR = [dict(n=(4, 64, 5)), dict(n=(5, 65, 4), slope_type=1), dict(n=(63, 4, 3), slope_type=0),
         dict(n=(250, 3, 3)), dict(n=(7, 130, 3), omega0=3.0)]


@pytest.mark.parametrize("case", range(len(SHEAR)))
def test_shearing_box_columns(case):
    kw = dict(SHEAR[case])
    pb = P.shearing_box(*kw.pop("n"), **kw)
    print(f"[gpu] shearing box columns, case {case}", flush=True)
    _same(pb, pb.params, 3)


# one tile of 33 columns, one of 34 (two of 17), 32 x 8, narrow tiles of 16
# rows, and planes that leave a short last block
VISC = [(32, 6, 5), (33, 7, 4), (31, 8, 9), (4, 33, 17), (65, 5, 3)]


@pytest.mark.parametrize("case", range(len(VISC)))
def test_viscous_tiles(case):
    pb = P.random_smooth(*VISC[case], seed=300 + case)
    p = pb.params.replace(nu=2e-3, eta=1e-3 if case % 2 else 0.0, iso=1 if case == 3 else 0,
                          ciso=1.0 if case == 3 else pb.params.ciso)
    print(f"[gpu] viscous tiles, case {case}", flush=True)
    _same(pb, p, 3)


# float64 launch shapes as created: one plane block under and over the line
# from which the fused kernel is taken (51 tiles of 17 x 5; 10 and 11 blocks of
# 4 planes), and tiles of which too few columns are used
@pytest.mark.parametrize("n", [(50, 84, 40), (50, 84, 43), (34, 100, 60), (84, 84, 172)])
def test_default_shape_gives_the_separate_kernels_bits(n):
    pb = P.random_smooth(*n, seed=sum(n))
    print(f"[gpu] default launch shape {n}", flush=True)
    a, b, c = (abi.Domain(pb.params, pb.uin) for _ in range(3))
    b.set_shape((0, 2), (0, 4))
    a.advance(2, 0.0)
    b.advance(2, 0.0)
    want = b.download()
    assert np.array_equal(a.download(), want)
    abi.Batch([c]).advance(2)   # keeps the separate kernels
    assert np.array_equal(c.download(), want)
    for d in (a, b, c):
        d.close()


# the forms that the default takes to the fused kernel: solvers, limiters,
# boundaries, isothermal, shear with and without FARGO, dissipation, the learned
# limiter
FORMS = [dict(riemann=P.HLL, riemann2d=P.LLF, slope_type=1), dict(riemann=P.LLF, riemann2d=P.UPWIND, slope_type=3),
         dict(riemann=P.UPWIND, riemann2d=P.HLLA, slope_type=0), dict(iso=1, ciso=1.0),
         dict(bdtype=(P.ZERO_GRADIENT, P.ZERO_GRADIENT, P.PERIODIC)), dict(nu=1e-3, eta=1e-3),
         dict(shear=0), dict(shear=1), dict(shear=0, iso=1, ciso=4e-2), dict(slope_type=4)]


@pytest.mark.parametrize("form", range(len(FORMS)))
def test_default_fused_form_gives_the_separate_kernels_bits(form):
    kw = dict(FORMS[form])
    n = (50, 84, 43)
    if "shear" in kw:
        pb = P.shearing_box(*n, fargo=kw.pop("shear"))
    else:
        pb = P.random_smooth(*n, seed=form)
    p = pb.params.replace(**kw)
    print(f"[gpu] default fused form {form}", flush=True)
    a, b = abi.Domain(p, pb.uin), abi.Domain(p, pb.uin)
    b.set_shape((0, 2), (0, 4))
    if p.slope_type == 4:
        for d in (a, b):
            d.set_limiter(learned.init_params(5))
    _, da = a.advance(2, 0.0)
    _, db = b.advance(2, 0.0)
    assert np.isfinite(da).all() and np.array_equal(da, db)
    assert np.array_equal(a.download(), b.download())
    for d in (a, b):
        d.close()


@pytest.mark.parametrize("precision", [0, 1])
def test_transfers_leave_the_run_unchanged(precision):
    """Downloads between steps change nothing, and an upload of a download
    goes on as the run does (its right faces are not read)."""
    pb = P.random_smooth(21, 6, 9, seed=77, precision=precision)
    print(f"[gpu] transfers, precision {precision}", flush=True)
    a, b = abi.Domain(pb.params, pb.uin), abi.Domain(pb.params, pb.uin)
    a.advance(1, 0.0)
    mid = a.download()
    a.advance(1)
    want = a.download()
    assert np.array_equal(want, a.download())
    mid[8:] = np.nan
    b.upload(mid)
    b.time = 0.0
    b.advance(1)
    assert np.array_equal(b.download(), want)
    for d in (a, b):
        d.close()
