"""The LDS-staged loop with every table in LDS, with the orbit and radii only,
with other parts and with none: the oracle's results bit for bit (the budget
caps make a plan of each kind for orbits of 601 and 3001 points)."""
import pytest

import frames
import oracle as orc
import fractalshades_amd as fsa
from gpu_util import run_gpu, assert_same

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("cap", [None, 130000, 75000, 61000, 50000, 20000])
@pytest.mark.parametrize("model,dx,max_iter", [("M2", "1e-100", 600), ("M2", "1e-12", 3000), ("M2", "1e-305", 3000),
                                               ("MN4", "1e-12", 3000), ("MN4", "1e-305", 3000), ("BS", "1e-12", 3000),
                                               ("BS", "1e-305", 3000)])
def test_shapes_bitexact(model, dx, max_iter, cap, monkeypatch):
    f = (fsa.Perturbation_mandelbrot(None) if model == "M2" else fsa.Perturbation_mandelbrot_N(None, 4)
         if model == "MN4" else fsa.Perturbation_burning_ship(None, "Burning ship"))
    f.zoom(precision=360, x={"M2": "-1.98", "MN4": "-1.25", "BS": "-1.9"}[model], y="0.", dx=dx, nx=26, xy_ratio=1.,
           theta_deg=0.)
    f.no_newton = True
    kw = dict(calc_name="t", subset=None, max_iter=max_iter, M_divergence=1.e3, BLA_eps=1.e-6)
    if f.holomorphic:
        kw.update(epsilon_stationnary=1.e-3, interior_detect=True, calc_dzndc=True)
    else:
        kw.update(calc_hessian=True)
    f.calc_std_div(**kw)
    args, c_pix = frames.frame_inputs(f)
    print(f"case {model} dx={dx} max_iter={max_iter} cap={cap}", flush=True)
    ref = orc.OracleCtx(args.fields, args.arrays).cycles(c_pix)
    assert 2 * ref[1].max() < len(args.arrays["Zn_path"])      # no pixel past the reference orbit's end
    if cap is not None:
        monkeypatch.setenv("FSG_LDS_BYTES", str(cap))
    got, _ = run_gpu(args, c_pix)
    assert_same(got, ref)
