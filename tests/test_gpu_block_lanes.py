"""A launch whose pixels are fewer than the chip's lanes runs in blocks of 256,
512 or 768 lanes: at the sizes where the block changes (256 CUs of one, two or
three waves per SIMD, one pixel less and more) the results and step counters
equal those of the kernel with its tables in global memory."""
import pytest

import frames
from gpu_util import run_gpu, assert_same

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", [0, 1], ids=["fp64", "fp32x"])
@pytest.mark.parametrize("n", [1, 257, 65536, 65537, 131073, 196607, 196609])
def test_block_lanes(n, precision, monkeypatch):
    f = frames.make("M2_int32", nx=450, max_iter=3000)
    args, c_pix = frames.frame_inputs(f)
    c_pix = c_pix[:n]
    args = args.with_fields(precision=precision)
    print(f"case M2_int32 npts={n} precision={precision}", flush=True)
    monkeypatch.delenv("FSG_TABLES", raising=False)
    got, stats = run_gpu(args, c_pix)
    assert c_pix.size == n
    monkeypatch.setenv("FSG_TABLES", "global")
    ref, ref_stats = run_gpu(args, c_pix)
    assert_same(got, ref)
    for key in ("plain_steps", "bla_steps", "bla_iters", "rebases", "bla_lookups", "redo_pixels"):
        assert stats[key] == ref_stats[key]
