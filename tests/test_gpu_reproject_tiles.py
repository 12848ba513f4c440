"""Depth reprojection at the edges of its 64x16 source tiles and of the 96x32
destination window a tile may take in LDS: partial tiles, shrinking and
stretching cameras (the stretched ones exceed the window and go to memory
directly), wild depths, several frames in a row. Bit-exact on millimetres."""
import numpy as np
import pytest

import hiprt
import oracle_lib as orc
import vscan

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("sw,sh,dw,dh", [(64, 16, 64, 16), (65, 17, 64, 16), (63, 15, 128, 96), (16, 16, 16, 16),
                                         (333, 251, 161, 117), (320, 240, 480, 360), (64, 48, 640, 480),
                                         (1, 1, 32, 32), (640, 480, 320, 240)])
def test_tiles(ctx, sw, sh, dw, dh):
    print(f"case: reprojection {sw}x{sh} -> {dw}x{dh}", flush=True)
    K = (0.8 * dw, 0.8 * dw, dw / 2 - 0.5, dh / 2 - 0.5)
    d = vscan.make_desc(vscan.WORKLOADS["plain_320x240_128"], n=16, W=dw, H=dh, K=K)
    s = vscan.Session(ctx, d)
    K_src = np.array([0.8 * sw, 0.8 * sw, sw / 2 - 0.5, sh / 2 - 0.5], np.float32)
    a = np.radians(3.0)
    T = np.array([[np.cos(a), -np.sin(a), 0, 0.03], [np.sin(a), np.cos(a), 0, -0.01], [0, 0, 1, 0.02], [0, 0, 0, 1]],
                 np.float32)
    rng = np.random.default_rng(sw * 7 + dw)
    src, dst = hiprt.DeviceBuffer(sw * sh * 2), hiprt.DeviceBuffer(dw * dh * 2)
    try:
        for k in range(3):
            y, x = np.mgrid[0:sh, 0:sw]
            mm = (900 + 2 * x + y + rng.integers(0, 30, (sh, sw))).astype(np.uint16)
            if k == 1:  # depths from nothing to everything: large windows
                mm = rng.integers(0, 65536, (sh, sw)).astype(np.uint16)
            mm[rng.random((sh, sw)) < 0.1] = 0
            if k == 2:
                mm[:] = 0  # no pixel lands
            src.upload(np.ascontiguousarray(mm))
            s.depth_reproject(src.ptr.value, sw, sh, K_src, T, dst_ptr=dst.ptr.value)
            s.sync()
            got = dst.download(np.zeros((dh, dw), np.uint16))
            want = orc.depth_reproject(mm, K_src, T, (dh, dw), np.float32(K))
            assert np.array_equal(got, want)
    finally:
        s.close()
        src.free()
        dst.free()
