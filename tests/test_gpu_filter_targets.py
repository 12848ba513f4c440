"""vs_bilateral_filter_depth into every kind of buffer that takes its result:
device memory, page-locked and pageable host memory, and device memory that is
not aligned to floats. The same bits as pyramid level 0, guard bytes untouched."""
import numpy as np
import pytest

import hiprt
import vscan

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("w,h", [(320, 240), (333, 251)])
@pytest.mark.parametrize("kind", ["device", "unaligned device", "page-locked", "pageable"])
def test_target(ctx, kind, w, h):
    print(f"case: filter {w}x{h} into {kind} memory", flush=True)
    st = vscan.SceneStream(3, seed=1, width=w, height=h)
    d = vscan.make_desc(vscan.WORKLOADS["plain_320x240_128"], n=32, W=w, H=h, K=st.K)
    s = vscan.Session(ctx, d)
    n, pad = w * h * 4, 64
    off = pad + (2 if kind.startswith("unaligned") else 0)
    dev = hiprt.DeviceBuffer(n + 2 * pad) if "device" in kind else None
    pin = hiprt.PinnedBuffer((n + 2 * pad,), np.uint8) if kind == "page-locked" else None
    host = pin.array if pin else np.zeros(n + 2 * pad, np.uint8)
    host[:] = 7
    try:
        if dev:
            dev.upload(host)
        base = dev.ptr.value if dev else host.ctypes.data
        frame = st.frame(1)
        vscan.check(vscan.lib().vs_bilateral_filter_depth(s.h, vscan._ptr(frame), 1, vscan.P(base + off), None),
                    "vs_bilateral_filter_depth")
        s.sync()
        got = dev.download(np.zeros(n + 2 * pad, np.uint8)) if dev else host
        want = s.filtered(0)
        assert (want > 0).any()
        assert got[off:off + n].tobytes() == want.tobytes()
        assert (got[:off] == 7).all() and (got[off + n:] == 7).all()
    finally:
        s.close()
        if dev:
            dev.free()
        if pin:
            pin.free()
