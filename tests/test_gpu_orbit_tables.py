"""calc_orbit with the tables in LDS and in global memory: the oracle's results
bit for bit for backshifts that divide the jumps' lengths, that jumps pass
several times over, and that are longer than a pixel's orbit."""
import pytest

import frames
import oracle as orc
import fractalshades_amd as fsa
from gpu_util import run_gpu, assert_same

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("tables", ["", "global"])
@pytest.mark.parametrize("model,dx", [("M2", "1e-12"), ("M2", "1e-305"), ("MN4", "1e-12"), ("MN4", "1e-305"),
                                      ("BS", "1e-12"), ("BS", "1e-305")])
@pytest.mark.parametrize("backshift", [1, 3, 8, 5000])
def test_orbit_bitexact(model, dx, backshift, tables, monkeypatch):
    f = (fsa.Perturbation_mandelbrot(None) if model == "M2" else fsa.Perturbation_mandelbrot_N(None, 4)
         if model == "MN4" else fsa.Perturbation_burning_ship(None, "Burning ship"))
    f.zoom(precision=360, x={"M2": "-1.98", "MN4": "-1.25", "BS": "-1.9"}[model], y="0.", dx=dx, nx=26, xy_ratio=1.,
           theta_deg=0.)
    f.no_newton = True
    kw = dict(calc_name="t", subset=None, max_iter=3000, M_divergence=1.e3, BLA_eps=1.e-6, calc_orbit=True,
              backshift=backshift)
    if f.holomorphic:
        kw.update(epsilon_stationnary=1.e-3, interior_detect=backshift != 3, calc_dzndc=True)
    else:
        kw.update(calc_hessian=True)
    f.calc_std_div(**kw)
    args, c_pix = frames.frame_inputs(f)
    print(f"case {model} dx={dx} backshift={backshift} tables={tables}", flush=True)
    ref = orc.OracleCtx(args.fields, args.arrays).cycles(c_pix)
    assert 2 * ref[1].max() < len(args.arrays["Zn_path"])      # no pixel past the reference orbit's end
    if tables:
        monkeypatch.setenv("FSG_TABLES", tables)
    got, _ = run_gpu(args, c_pix)
    assert_same(got, ref)
