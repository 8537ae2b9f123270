"""The z^d + c kernels with their tables in LDS are compiled for dz/dc alone,
for both derivatives, and once more reading the combination from the launch
arguments: each combination against the oracle, binary64 and extended range,
for the lowest, a middle and the highest degree."""
import pytest

import frames
import oracle as orc
from gpu_util import run_gpu, assert_same
from fractalshades_amd.perturbation import CycleIndepArgs

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("d", [3, 5, 8])
@pytest.mark.parametrize("dc,dz", [(0, 0), (1, 0), (0, 1), (1, 1)])
@pytest.mark.parametrize("xr", [0, 1])
def test_mn_derivative_combinations_bitexact(d, dc, dz, xr):
    f = frames.mn_frame(d, nx=40)
    args, c_pix = frames.frame_inputs(f)
    args = CycleIndepArgs(dict(args.fields, calc_dzndc=dc, interior_detect=dz, xr_mode=xr), args.arrays, None,
                          projection=args.projection)
    print(f"case MN d={d} dc={dc} dz={dz} xr={xr} npts={c_pix.size}", flush=True)
    ref = orc.OracleCtx(args.fields, args.arrays).cycles(c_pix)
    got, stats = run_gpu(args, c_pix)
    assert_same(got, ref)
    assert stats["plain_steps"] > 0
