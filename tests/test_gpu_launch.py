"""Launch shapes at the ends of the accepted domain sizes, and as created."""
import numpy as np
import pytest

from dmx import abi
from dmx import learned
from dmx import problems as P
from test_gpu_columns import FORMS

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


# float64 boxes as created: thin ones and few tiles keep the separate kernels
KEPT = {(224, 224, 4): "flux", (50, 84, 43): "flux", (101, 50, 37): "flux", (64, 64, 64): "fused",
        (30, 92, 225): "fused"}


@pytest.mark.parametrize("n", list(KEPT))
def test_default_kernels(n):
    pb = P.random_smooth(*n, seed=sum(n))
    print(f"[gpu] default kernels {n}", flush=True)
    a, b = abi.Domain(pb.params, pb.uin), abi.Domain(pb.params, pb.uin)
    ms = a.profile(2, 0.0)
    assert (ms["fused"] > 0.0) == (KEPT[n] == "fused") and (ms["flux"] > 0.0) == (KEPT[n] == "flux"), ms
    b.set_shape((3, 4) if KEPT[n] == "flux" else (0, 2), (0, 4))   # the other form
    b.advance(2, 0.0)
    assert np.array_equal(a.download(), b.download())
    for d in (a, b):
        d.close()


@pytest.mark.parametrize("form", range(len(FORMS)))
def test_default_fused_forms(form):
    """The forms of test_gpu_columns on a box whose default is the fused kernel."""
    kw = dict(FORMS[form])
    n = (64, 64, 64)
    pb = P.shearing_box(*n, fargo=kw.pop("shear")) if "shear" in kw else P.random_smooth(*n, seed=form)
    p = pb.params.replace(**kw)
    print(f"[gpu] default fused form {form}", flush=True)
    a, b = abi.Domain(p, pb.uin), abi.Domain(p, pb.uin)
    b.set_shape((0, 2), (0, 4))
    if p.slope_type == 4:
        for d in (a, b):
            d.set_limiter(learned.init_params(5))
    assert a.profile(2, 0.0)["fused"] > 0.0
    b.advance(2, 0.0)
    assert np.array_equal(a.download(), b.download())
    for d in (a, b):
        d.close()
