"""Escape and interior tests at the ends of their parameters' ranges, where a
filter taken by one component decides first: the oracle's results bit for bit
for escape radii from 2 to 1e100 and stationarity bounds from loose to one
whose square underflows, binary64 and extended-range deltas."""
import numpy as np
import pytest

import frames
import oracle as orc
import fractalshades_amd as fsa
from gpu_util import run_gpu, assert_same
from fractalshades_amd.perturbation import CycleIndepArgs

pytestmark = pytest.mark.gpu


def frame(model, dx):
    f = (fsa.Perturbation_mandelbrot(None) if model == "M2" else fsa.Perturbation_mandelbrot_N(None, 4)
         if model == "MN4" else fsa.Perturbation_burning_ship(None, "Burning ship"))
    x = {"M2": "-1.98", "MN4": "-1.25", "BS": "-1.9"}[model]
    f.zoom(precision=360, x=x, y="0.", dx=dx, nx=32, xy_ratio=1., theta_deg=0.)
    f.no_newton = True
    kw = dict(calc_name="t", subset=None, max_iter=3000, M_divergence=1.e3, BLA_eps=1.e-6)
    if f.holomorphic:
        kw.update(epsilon_stationnary=1.e-3, interior_detect=True, calc_dzndc=True)
    else:
        kw.update(calc_hessian=True)
    f.calc_std_div(**kw)
    return f


@pytest.mark.parametrize("model,dx", [("M2", "5e-2"), ("M2", "1e-12"), ("M2", "1e-305"), ("MN4", "5e-2"),
                                      ("MN4", "1e-305"), ("BS", "5e-2"), ("BS", "1e-305")])
@pytest.mark.parametrize("radius,eps", [(2., 0.5), (1.e3, 1.e-170), (2.**31, 1.e-3), (1.e100, 0.)])
def test_stop_tests_bitexact(model, dx, radius, eps):
    args, c_pix = frames.frame_inputs(frame(model, dx))
    fields = dict(args.fields, M_divergence=radius, epsilon_stationnary=eps)
    args = CycleIndepArgs(fields, args.arrays, None, projection=args.projection)
    print(f"case {model} dx={dx} radius={radius} eps={eps} xr={fields['xr_mode']}", flush=True)
    ref = orc.OracleCtx(args.fields, args.arrays).cycles(c_pix)
    assert 2 * ref[1].max() < len(args.arrays["Zn_path"])  # no pixel past the reference orbit's end
    got, _ = run_gpu(args, c_pix)
    for Z in (got[0], ref[0]):                  # an overflown pixel's NaNs have no sign
        v = Z.view(np.float64)
        v[np.isnan(v)] = np.nan
    assert_same(got, ref)
