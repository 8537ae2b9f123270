"""Extended-range kernels on frames centred on the real axis, where orbit
points have a zero imaginary part, the deltas' binary64 copies underflow and
the pixels of the middle row and column have a zero coordinate: the oracle's
results bit for bit, for every model and burning-ship flavour."""
import numpy as np
import pytest

import frames
import oracle as orc
import fractalshades_amd as fsa
from gpu_util import run_gpu, assert_same
from fractalshades_amd.models import BS_FLAVORS
from fractalshades_amd.perturbation import CycleIndepArgs

pytestmark = pytest.mark.gpu
MODELS = ["M2", "MN3", "MN4", "MN6"] + list(BS_FLAVORS)


# on the set's real antenna (but for the middle row, which never escapes, the
# pixels escape after about 1000 iterations), or inside the set
CENTRES = {"M2": "-1.98", "MN3": "0.3849", "MN4": "-1.25", "MN6": "-1.1"}


def frame(model, dx, nx):
    x = CENTRES.get(model, "-1.9")
    if model == "M2":
        f = fsa.Perturbation_mandelbrot(None)
    elif model.startswith("MN"):
        f = fsa.Perturbation_mandelbrot_N(None, int(model[2:]))
    else:
        f = fsa.Perturbation_burning_ship(None, model)
    f.zoom(precision=360, x=x, y="0.", dx=dx, nx=nx, xy_ratio=1., theta_deg=0.)
    f.no_newton = True
    kw = dict(calc_name="t", subset=None, max_iter=3000, M_divergence=1.e3, BLA_eps=1.e-6)
    if f.holomorphic:
        kw.update(epsilon_stationnary=1.e-3, interior_detect=True, calc_dzndc=True)
    else:
        kw.update(calc_hessian=True)
    f.calc_std_div(**kw)
    return f


# BLA on: frames without a middle row or column for the antenna's holomorphic
# models (a pixel that stays on it would run past the orbit's end)
CASES = [(m, 0, 33) for m in MODELS] + [(m, 1, 33) for m in BS_FLAVORS] + [("M2", 1, 32), ("MN4", 1, 32)]


@pytest.mark.parametrize("model,bla,nx", CASES)
@pytest.mark.parametrize("dx", ["1e-305", "1e-330"])
def test_real_axis_bitexact(model, dx, bla, nx):
    f = frame(model, dx, nx)
    args, c_pix = frames.frame_inputs(f)
    args = CycleIndepArgs(dict(args.fields, bla_on=bla), args.arrays, None, projection=args.projection)
    print(f"case {model} dx={dx} bla={bla} xr={args.fields['xr_mode']} npts={c_pix.size}", flush=True)
    assert args.fields["xr_mode"] == 1
    ref = orc.OracleCtx(args.fields, args.arrays).cycles(c_pix)
    got, stats = run_gpu(args, c_pix)
    assert stats["plain_steps"] > 0
    assert_same(got, ref)
