"""In-place vertex / normal maps of one session and level on two streams at
once, into different buffers: the calls share nothing, so every pair of maps is
the one a call alone writes. Buffers of odd widths start their rows at every
4-byte alignment."""
import numpy as np
import pytest

import hiprt
import vscan
from test_gpu_normals_order import ramps

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("w,h,level", [(640, 480, 0), (1281, 721, 0), (643, 481, 1), (67, 49, 2), (8192, 40, 0)])
def test_two_streams(ctx, w, h, level):
    print(f"case: in-place maps of level {level} of {w}x{h} on two streams", flush=True)
    d = vscan.make_desc(vscan.WORKLOADS["plain_320x240_128"], n=16, W=w, H=h, K=(400.0, 400.0, w / 2, h / 2))
    s = vscan.Session(ctx, d)
    lw, lh = w >> level, h >> level
    n = lw * lh * 3
    streams = [hiprt.Stream() for _ in range(2)]
    pad = 64  # bytes around each map that stay as they are
    bufs = [[hiprt.DeviceBuffer(n * 4 + 2 * pad) for _ in range(2)] for _ in range(2)]
    try:
        s.set_filtered(level, ramps(lh, lw, 5))

        def fill():
            for pair in bufs:
                for b in pair:
                    b.upload(np.full(n + 2 * pad // 4, 7.0, np.float32))

        def call(k):
            v, m = (vscan.P(b.ptr.value + pad) for b in bufs[k])
            vscan.check(vscan.lib().vs_vertex_normal_maps_inplace(s.h, level, v, m, streams[k].h), "vnmap inplace")

        def read(k):
            streams[k].sync()
            return [b.download(np.zeros(n + 2 * pad // 4, np.float32)) for b in bufs[k]]

        fill()
        call(0)
        want = read(0)
        for m in want:
            assert (m[:pad // 4] == 7.0).all() and (m[-pad // 4:] == 7.0).all()
        assert (want[0] == -100.0).any() and (want[1] != -100.0).any()
        for _ in range(8):
            fill()
            for _ in range(5):
                call(0)
                call(1)
            for k in range(2):
                for a, b in zip(read(k), want):
                    assert np.array_equal(a, b)
    finally:
        for x in streams:
            x.sync()
            x.destroy()
        for pair in bufs:
            for b in pair:
                b.free()
        s.close()
