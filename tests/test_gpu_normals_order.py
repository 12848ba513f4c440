"""In-place vertex / normal maps at the edges of their bit rows: frame widths
around one, two and many 64-pixel words, and around the 4096 columns where a
lane of the ordering wave takes a second word. Runs of grazing pixels of every
length cross words, lanes and whole rows.

Masks are bit-exact against the oracle's in-place loop; values within the
FP32 rounding of a back-projection (1e-6 relative) and of a normal (1e-5).
"""
import numpy as np
import pytest

import hiprt
import oracle_lib as orc
import vscan

pytestmark = pytest.mark.gpu


def ramps(h, w, seed):
    """Depth of flat and steep column blocks of random lengths, redrawn every
    few rows, with some invalid pixels: gradients are 0 or far above the
    grazing limit, so FP32 and FP64 agree on every mask."""
    rng = np.random.default_rng(seed)
    z = np.zeros((h, w), np.float32)
    y = 0
    while y < h:
        rows = int(rng.integers(1, 9))
        step, x = np.zeros(w), 0
        while x < w:
            n = int(rng.choice([1, 2, 3, 7, 63, 64, 65, 130, w]))
            step[x:x + n] = rng.choice([0.0, 0.05, -0.05]) * (1 if n < 200 else 0.2)
            x += n
        z[y:y + rows] = 1.5 + 0.9 * np.abs((np.cumsum(step) / 0.9 + 1) % 2 - 1)
        y += rows
    z[rng.random((h, w)) < 0.02] = 0.0
    return z


@pytest.mark.parametrize("w,h", [(16, 16), (63, 20), (64, 17), (65, 33), (128, 40), (640, 50), (4096, 20), (4097, 18),
                                 (8192, 17)])
def test_order_at_word_edges(ctx, w, h):
    print(f"case: in-place maps {w}x{h}", flush=True)
    d = vscan.make_desc(vscan.WORKLOADS["plain_320x240_128"], n=16, W=w, H=h, K=(400.0, 400.0, w / 2, h / 2))
    s = vscan.Session(ctx, d)
    try:
        for seed in (1, 2):
            z = ramps(h, w, seed)
            s.set_filtered(0, z)
            v, n = hiprt.DeviceBuffer(h * w * 12), hiprt.DeviceBuffer(h * w * 12)
            try:
                vscan.check(vscan.lib().vs_vertex_normal_maps_inplace(s.h, 0, v.ptr, n.ptr, None), "vnmap inplace")
                s.sync()
                gv = v.download(np.zeros((h, w, 3), np.float32))
                gn = n.download(np.zeros((h, w, 3), np.float32))
            finally:
                v.free()
                n.free()
            rv, rn = orc.vnmap(z, orc.K_levels(d)[0], inplace=True)
            assert np.array_equal(gv[..., 0] == -100, rv[..., 0] == -100)
            assert np.array_equal(gn[..., 0] == -100, rn[..., 0] == -100)
            grazing = int(((rv[..., 0] == -100) & (z > 0)).sum())
            assert grazing > h, "the frame has runs of grazing pixels"
            np.testing.assert_allclose(gv, rv, rtol=1e-6, atol=1e-6)
            np.testing.assert_allclose(gn, rn, rtol=0, atol=1e-5)
    finally:
        s.close()
