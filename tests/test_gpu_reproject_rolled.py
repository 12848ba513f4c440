"""Depth reprojection between cameras rolled against each other: a tile's
destination window is then as high as it is wide, or a column, and at the edge
of what the window takes in one band of 4096 pixels, in four, and beyond. Bit-exact on millimetres."""
import numpy as np
import pytest

import hiprt
import oracle_lib as orc
import vscan

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("scale", [0.5, 1.0, 1.12, 1.15, 2.0, 3.0])  # at 45 degrees (57 scale)^2 pixels: 1 to 4 bands, then none
@pytest.mark.parametrize("deg", [35.0, 45.0, 90.0, 180.0, -120.0])
def test_rolled(ctx, deg, scale):
    print(f"case: cameras rolled by {deg} degrees, scale {scale}", flush=True)
    sw, sh = 321, 243
    dw = dh = int(340 * scale)
    K_src = np.array([260.0, 260.0, sw / 2 - 0.5, sh / 2 - 0.5], np.float32)
    K = (260.0 * scale, 260.0 * scale, dw / 2 - 0.5, dh / 2 - 0.5)
    d = vscan.make_desc(vscan.WORKLOADS["plain_320x240_128"], n=16, W=dw, H=dh, K=K)
    s = vscan.Session(ctx, d)
    a = np.radians(deg)
    T = np.array([[np.cos(a), -np.sin(a), 0, 0.01], [np.sin(a), np.cos(a), 0, -0.01], [0, 0, 1, 0.0], [0, 0, 0, 1]],
                 np.float32)
    rng = np.random.default_rng(int(abs(deg)) * 10 + int(scale * 100))
    y, x = np.mgrid[0:sh, 0:sw]
    src, dst = hiprt.DeviceBuffer(sw * sh * 2), hiprt.DeviceBuffer(dw * dh * 2)
    try:
        for _ in range(2):
            mm = (900 + 2 * x + y + rng.integers(0, 30, (sh, sw))).astype(np.uint16)
            mm[rng.random((sh, sw)) < 0.1] = 0
            src.upload(np.ascontiguousarray(mm))
            s.depth_reproject(src.ptr.value, sw, sh, K_src, T, dst_ptr=dst.ptr.value)
            s.sync()
            got = dst.download(np.zeros((dh, dw), np.uint16))
            want = orc.depth_reproject(mm, K_src, T, (dh, dw), np.float32(K))
            assert (want > 0).sum() > 1000
            assert np.array_equal(got, want)
    finally:
        s.close()
        src.free()
        dst.free()
