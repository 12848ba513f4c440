"""Large downloads (from 16 MB on, where pageable host memory goes through the
staging lanes) into page-locked and device memory, alone and mixed with
pageable memory in one call, and snapshots and colours into page-locked memory:
the same bytes as into pageable memory."""
import ctypes as C

import numpy as np
import pytest

import hiprt
import vscan

pytestmark = pytest.mark.gpu


def volume(dims, seed):
    rng = np.random.default_rng(seed)
    return (rng.uniform(-1, 1, dims[::-1]).astype(np.float32), rng.integers(0, 100, dims[::-1]).astype(np.float32))


def session(ctx, dims, color=False):
    d = vscan.make_desc(vscan.WORKLOADS["plain_320x240_128"], n=64, W=64, H=48, K=(60.0, 60.0, 31.5, 23.5),
                        integrate_mode=vscan.VS_INTEGRATE_COLOR if color else vscan.VS_INTEGRATE_DEPTH)
    for k in range(3):
        d.vol_dim[k] = dims[k]
    return vscan.Session(ctx, d)


class Pageable:
    def __init__(self, shape):
        self.array = np.zeros(shape, np.float32)
        self.ptr = vscan._ptr(self.array)

    def read(self):
        return self.array

    def free(self):
        pass


class Pinned(Pageable):
    def __init__(self, shape):
        self.buf = hiprt.PinnedBuffer(shape, np.float32)
        self.array, self.ptr = self.buf.array, self.buf.ptr

    def free(self):
        self.array = None
        self.buf.free()


class Device(Pageable):
    def __init__(self, shape):
        self.shape = shape
        self.buf = hiprt.DeviceBuffer(int(np.prod(shape)) * 4)
        self.ptr = self.buf.ptr

    def read(self):
        return self.buf.download(np.zeros(self.shape, np.float32))

    def free(self):
        self.buf.free()


@pytest.mark.parametrize("dims", [(128, 128, 120), (200, 136, 168)])  # below and above the lanes' limit
@pytest.mark.parametrize("to", [(Pinned, Pinned), (Device, Device), (Pageable, Pinned), (Device, Pageable)])
def test_volume(ctx, dims, to):
    print(f"case: download of {dims} into {[t.__name__ for t in to]}", flush=True)
    s = session(ctx, dims)
    F, W = volume(dims, 3)
    f, w = to[0](F.shape), to[1](W.shape)
    try:
        s.set_volume(F, W)
        for _ in range(2):
            vscan.check(vscan.lib().vs_volume_download(s.h, f.ptr, w.ptr, None), "vs_volume_download")
            assert np.array_equal(f.read(), F) and np.array_equal(w.read(), W)
    finally:
        f.free()
        w.free()
        s.close()


def test_snapshot_and_colour(ctx):
    dims = (200, 136, 168)
    print("case: snapshot and colour volume into page-locked memory", flush=True)
    s = session(ctx, dims, color=True)
    bufs = []
    try:
        s.set_volume(*volume(dims, 4))
        want = s.snapshot()
        assert len(want) > 16 << 20
        snap = hiprt.PinnedBuffer((len(want),), np.uint8)
        bufs.append(snap)
        n = C.c_size_t()
        vscan.check(vscan.lib().vs_session_snapshot(s.h, snap.ptr, len(want), C.byref(n)), "vs_session_snapshot")
        assert n.value == len(want) and snap.array.tobytes() == want
        rgb = s.volume_color()
        pin = hiprt.PinnedBuffer(rgb.shape, np.uint8)
        bufs.append(pin)
        pin.array[:] = 9
        vscan.check(vscan.lib().vs_volume_download_color(s.h, pin.ptr), "vs_volume_download_color")
        assert np.array_equal(pin.array, rgb)
    finally:
        for b in bufs:
            b.free()
        s.close()
