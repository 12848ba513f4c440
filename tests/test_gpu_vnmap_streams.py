"""In-place vertex / normal maps of one session and level on two streams at
once, two of the caller's or the session's own and one of the caller's, and from
two threads on the session's own, into different buffers: every pair of maps is
the one a call alone writes. Rows of odd widths start at every 4-byte
alignment."""
import threading

import numpy as np
import pytest

import hiprt
import vscan
from test_gpu_normals_order import ramps

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("own", [False, True])
@pytest.mark.parametrize("w,h,level", [(640, 480, 0), (1281, 721, 0), (643, 481, 1), (67, 49, 2), (8192, 40, 0)])
def test_two_streams(ctx, w, h, level, own):
    print(f"case: in-place maps of level {level} of {w}x{h} on two streams, own: {own}", flush=True)
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
            vscan.check(vscan.lib().vs_vertex_normal_maps_inplace(s.h, level, v, m, None if own and k == 0 else streams[k].h), "vnmap inplace")

        def read(k):
            streams[k].sync()
            s.sync()
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


def test_two_threads(ctx):
    w, h = 641, 482
    print("case: in-place maps from two threads on the session's own stream", flush=True)
    d = vscan.make_desc(vscan.WORKLOADS["plain_320x240_128"], n=16, W=w, H=h, K=(400.0, 400.0, w / 2, h / 2))
    s = vscan.Session(ctx, d)
    bufs = [[hiprt.DeviceBuffer(w * h * 12) for _ in range(2)] for _ in range(3)]
    try:
        s.set_filtered(0, ramps(h, w, 5))

        def work(k, n):
            for _ in range(n):
                vscan.check(vscan.lib().vs_vertex_normal_maps_inplace(s.h, 0, bufs[k][0].ptr, bufs[k][1].ptr, None),
                            "vnmap inplace")

        work(2, 1)
        threads = [threading.Thread(target=work, args=(k, 200)) for k in range(2)]
        for t in threads:
            t.start()
        for t in threads:
            t.join()
        s.sync()
        want = [b.download(np.zeros((h, w, 3), np.float32)) for b in bufs[2]]
        for pair in bufs[:2]:
            for b, m in zip(pair, want):
                assert np.array_equal(b.download(np.zeros((h, w, 3), np.float32)), m)
    finally:
        s.sync()
        for pair in bufs:
            for b in pair:
                b.free()
        s.close()
