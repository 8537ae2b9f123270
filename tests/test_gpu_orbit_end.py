"""Pixels that follow an orbit without escape or period to its last point by a
jump and end on the point after it: the whole numbers and derivatives of the
oracle, which is given that point (an orbit longer by one), in every
arrangement of the tables."""
import numpy as np
import pytest

import frames
import oracle as orc
import fractalshades_amd as fsa
from gpu_util import run_gpu

MAX_ITER = 600           # a multiple of 8: a jump can end on the last point, 600
DEGREE = {"M2": 2, "MN4": 4, "BS": 2}
CASES = [(m, dx) for m in DEGREE for dx in ("1e-12", "1e-305")]


def _model(model):
    return (fsa.Perturbation_mandelbrot(None) if model == "M2" else fsa.Perturbation_mandelbrot_N(None, 4)
            if model == "MN4" else fsa.Perturbation_burning_ship(None, "Burning ship"))


def _frame(model, dx, orbit=None, **over):
    f = _model(model)
    f.zoom(precision=330, x="-0.1", y="0.15", dx=dx, nx=20, xy_ratio=1., theta_deg=0.)
    f.no_newton = True
    kw = dict(calc_name="t", subset=None, max_iter=MAX_ITER, M_divergence=1.e3, BLA_eps=1.e-6)
    if f.holomorphic:
        kw.update(epsilon_stationnary=1.e-3, interior_detect=False, calc_dzndc=True)
    else:
        kw.update(calc_hessian=True)
    kw.update(over)
    if orbit is not None:
        f.max_iter = kw["max_iter"]
        f.set_reference(*orbit)
    f.calc_std_div(**kw)
    return f


def _longer(f, model, dx):
    """The oracle's inputs: f's own, with the orbit's next point."""
    args, c_pix = frames.frame_inputs(f)
    g = _frame(model, dx, max_iter=MAX_ITER + 1)
    longer = frames.frame_inputs(g)[0]
    Zn = longer.arrays["Zn_path"]
    assert np.array_equal(Zn[:-2], args.arrays["Zn_path"])
    assert args.fields["ref_div_iter"] == args.fields["ref_len"] == MAX_ITER + 1           # no escape
    fields = dict(args.fields, ref_len=MAX_ITER + 2, ref_div_iter=MAX_ITER + 2)
    return args, c_pix, fields, dict(args.arrays, Zn_path=Zn)


@pytest.mark.parametrize("model,dx", CASES)
def test_case_reaches_the_entry(model, dx):
    args, c_pix, fields, arrays = _longer(_frame(model, dx), model, dx)
    _, U, sr, si = orc.OracleCtx(fields, arrays).cycles(c_pix)
    # (the burning-ship loop keeps the index of the step's start when max_iter stops it)
    assert (U == (MAX_ITER if model == "BS" else MAX_ITER + 1)).all()
    assert (si == MAX_ITER + 1).all() and (sr == 0).all()


@pytest.mark.gpu
@pytest.mark.parametrize("tables", ["lds", "part", "global"])
@pytest.mark.parametrize("precision", ["fp64", "fp32x"])
@pytest.mark.parametrize("model,dx", CASES)
def test_results_at_the_orbit_end(model, dx, precision, tables, monkeypatch):
    print(f"case {model} dx={dx} {precision} {tables}", flush=True)
    args, c_pix, fields, arrays = _longer(_frame(model, dx), model, dx)
    want = orc.OracleCtx(fields, arrays).cycles(c_pix)
    if tables == "part":
        monkeypatch.setenv("FSG_LDS_BYTES", "16000")
    if tables == "global":
        monkeypatch.setenv("FSG_TABLES", "global")
    if precision == "fp32x":
        args = args.with_fields(precision=1)
    got, _ = run_gpu(args, c_pix)
    for a, b in zip(got[1:], want[1:]):
        np.testing.assert_array_equal(a, b)
    Z, W = got[0], want[0]
    rows = 2 if model == "BS" else 1
    # Z_L from the rounded Z_{L-1}: f' times half an ulp of it, d + 1 roundings of
    # values of modulus <= 2 (4 for both parts); binary32 adds 2^-20 of z, here below
    tol = 4 * (DEGREE[model] * 2. ** (DEGREE[model] - 1) + DEGREE[model] + 1) * 2.**-53
    assert np.abs(W[:rows]).max() < 2.
    np.testing.assert_allclose(Z[:rows], W[:rows], rtol=0., atol=tol)
    if precision == "fp64":
        np.testing.assert_array_equal(Z[rows:].view(np.uint64), W[rows:].view(np.uint64))
    else:
        scale = np.abs(W[rows:]).max()
        np.testing.assert_allclose(Z[rows:], W[rows:], rtol=0., atol=1.e-4 * scale)


@pytest.mark.gpu
def test_longer_max_iter_than_the_orbit():
    """An orbit shorter than the period given for it, and a max_iter past it:
    pixels rebase at its last point, as with no period given."""
    f = _frame("M2", "1e-12")
    p = f.FP_params
    orbit = (p["ref_point"], None, f.Zn_path, len(f.Zn_path), p["xr"])
    frame = [_frame("M2", "1e-12", orbit=(orbit[0], order, *orbit[2:]), max_iter=2000) for order in (None, 5000)]
    got = []
    for g in frame:
        args, c_pix = frames.frame_inputs(g)
        assert args.fields["ref_div_iter"] == (len(f.Zn_path) if g is frame[0] else 2001)
        got.append(run_gpu(args, c_pix)[0])
    for a, b in zip(*got):
        np.testing.assert_array_equal(a, b)
