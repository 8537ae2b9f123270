"""Wide frames around short reference orbits, binary64 deltas: pixels rebase at
every few steps, at a last orbit point reached right after a rebase too, or
follow a cycle of three points over its end.  The oracle's results bit for
bit, for each combination of derivatives and with the orbit recorder."""
import numpy as np
import pytest

import frames
import oracle as orc
from fractalshades_amd.perturbation import REF_ORDER_NONE, CycleIndepArgs
from gpu_util import assert_same, run_gpu

# name: (reference point, orbit points, first invalid index, order)
ORBITS = {
    "div3": (0.6 + 0.6j, 8, 3, None),
    "div4": (0.6 + 0.6j, 8, 4, None),
    "div5": (-0.5 + 0.5j, 9, 5, None),
    "to_its_end": (-0.5 + 0.5j, 40, 40, None),
    "cycle3": (-1.7548776662466927 + 0j, 3, None, 3),
    "cycle3_cut": (-1.7548776662466927 + 0j, 3, 3, 3),
}
MAX_ITER = 400


def inputs(orbit, degree, dz, dc, backshift):
    ref, L, div, order = ORBITS[orbit]
    f = (frames.make("M2_E11", nx=24, interior_detect=True, calc_dzndc=True) if degree == 2
         else frames.mn_frame(degree, nx=24))
    args, c_pix = frames.frame_inputs(f)
    Zn = np.zeros(L, np.complex128)
    for i in range(1, L):
        Zn[i] = Zn[i - 1] ** degree + ref if abs(Zn[i - 1]) < 1e3 else 0.
    drift = -0.4 - ref
    fields = dict(args.fields, ref_len=L, ref_div_iter=MAX_ITER + 1 if div is None else div,
                  ref_order=REF_ORDER_NONE if order is None else order, dx_mant=1.5, dx_exp=1, bla_on=0,
                  drift_mant=(drift.real, drift.imag), drift_exp=(0, 0), kc_mant=1., kc_exp=2, max_iter=MAX_ITER,
                  calc_dzndc=int(dc), interior_detect=int(dz), calc_orbit=int(backshift > 0), backshift=backshift)
    arrays = dict(args.arrays, Zn_path=Zn.view(np.float64).copy(), xr_index=np.zeros(0, np.int32),
                  xr_mant=np.zeros(0), xr_exp=np.zeros(0, np.int32))
    return CycleIndepArgs(fields, arrays, args.interrupted), c_pix


@pytest.mark.gpu
@pytest.mark.parametrize("tables", ["lds", "global"])
@pytest.mark.parametrize("degree,dz,dc,backshift", [(2, 1, 1, 0), (2, 0, 1, 0), (2, 1, 0, 0), (2, 0, 0, 0), (2, 1, 1, 2),
                                                    (3, 1, 1, 0), (3, 0, 1, 0), (3, 1, 1, 3), (3, 0, 1, 3), (3, 1, 0, 3)])
@pytest.mark.parametrize("orbit", sorted(ORBITS))
def test_bitexact(orbit, degree, dz, dc, backshift, tables, monkeypatch):
    print(f"case {orbit} d={degree} dz={dz} dc={dc} backshift={backshift} {tables}", flush=True)
    args, c_pix = inputs(orbit, degree, dz, dc, backshift)
    want = orc.OracleCtx(args.fields, args.arrays).cycles(c_pix)
    if tables == "global":
        monkeypatch.setenv("FSG_TABLES", "global")
    got, stats = run_gpu(args, c_pix)
    assert_same(got, want)
    assert stats["rebases"] > 0


@pytest.mark.parametrize("orbit", sorted(ORBITS))
def test_frames_hold_escaping_and_bounded_pixels(orbit):
    args, c_pix = inputs(orbit, 2, 0, 1, 0)
    _, U, sr, si = orc.OracleCtx(args.fields, args.arrays).cycles(c_pix)
    assert (sr == 1).any() and (sr == 0).any() and len(np.unique(si)) > 5
    assert U.max() < args.fields["ref_len"]
