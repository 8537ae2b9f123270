"""Results of host-buffer tiles through the pinned buffers: tiles from one pixel
to past the largest buffer, on contexts that come and go and from several
threads at once, equal the static-staging entry point's bit for bit, step
counters included."""
import threading

import numpy as np
import pytest

import frames
from gpu_util import run_gpu, assert_same

pytestmark = pytest.mark.gpu


def _alone(args, c_pix):
    n = c_pix.size
    out = (np.zeros((2, n), np.complex128), np.zeros((1, n), np.int32), -np.ones((1, n), np.int8),
           np.zeros((1, n), np.int32))
    rc, st = args.ctx.tile(c_pix, *out, noalloc=True)
    assert rc == 0
    return out, st


def _inputs():
    return frames.frame_inputs(frames.make("M2_E20", nx=640, max_iter=20000))


@pytest.mark.parametrize("n", [1, 63, 4097, 40000, 409000, 409600])
def test_sizes(n):
    args, c_pix = _inputs()
    c = np.ascontiguousarray(c_pix[:n])
    got, st = run_gpu(args, c)
    want, st_want = _alone(args, c[:40000])
    assert_same(tuple(np.ascontiguousarray(x[:, :40000]) for x in got), want)
    if n <= 40000:
        assert {k: v for k, v in st.items() if k != "kernel_ms"} == {k: v for k, v in st_want.items() if k != "kernel_ms"}


def test_threads_and_contexts():
    args, c_pix = _inputs()
    want = [_alone(args, np.ascontiguousarray(c_pix[k::8]))[0] for k in range(8)]
    bad = []

    def run(k):
        for _ in range(3):
            own = args.with_fields(max_iter=20000)          # a context of its own, given up after the tile
            got, _ = run_gpu(own, np.ascontiguousarray(c_pix[k::8]))
            try:
                assert_same(got, want[k])
            except AssertionError as e:
                bad.append((k, str(e)))

    threads = [threading.Thread(target=run, args=(k,)) for k in range(8)]
    for t in threads:
        t.start()
    for t in threads:
        t.join(timeout=60)
    assert not any(t.is_alive() for t in threads) and not bad
