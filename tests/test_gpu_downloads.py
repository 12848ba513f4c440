"""Volume downloads around the size from which they go through the staging
lanes (16 MB), with partial last pieces, from several threads of one context
at once, against the uploaded volume."""
import threading

import numpy as np
import pytest

import vscan

pytestmark = pytest.mark.gpu


def make(ctx, dims, seed):
    d = vscan.make_desc(vscan.WORKLOADS["plain_320x240_128"], n=64, W=64, H=48, K=(60.0, 60.0, 31.5, 23.5))
    for k in range(3):
        d.vol_dim[k] = dims[k]
    s = vscan.Session(ctx, d)
    rng = np.random.default_rng(seed)
    F = rng.uniform(-1, 1, dims[::-1]).astype(np.float32)
    W = rng.integers(0, 100, dims[::-1]).astype(np.float32)
    s.set_volume(F, W)
    return s, F, W


@pytest.mark.parametrize("dims", [(128, 128, 120), (128, 128, 128), (128, 128, 136), (200, 136, 168)])
def test_sizes(ctx, dims):
    print(f"case: download of {dims}", flush=True)
    s, F, W = make(ctx, dims, 1)
    try:
        for _ in range(2):
            gF, gW, _ = s.volume()
            assert np.array_equal(gF, F) and np.array_equal(gW, W)
        only = np.zeros_like(F)
        vscan.check(vscan.lib().vs_volume_download(s.h, None, vscan._ptr(only), None), "vs_volume_download")
        assert np.array_equal(only, W)
    finally:
        s.close()


def test_threads(ctx):
    print("case: downloads of three sessions from three threads", flush=True)
    made = [make(ctx, (136, 128, 136), k) for k in range(3)]
    bad = []

    def work(s, F, W):
        for _ in range(3):
            gF, gW, _ = s.volume()
            if not (np.array_equal(gF, F) and np.array_equal(gW, W)):
                bad.append(s)

    try:
        t = [threading.Thread(target=work, args=m) for m in made]
        for x in t:
            x.start()
        for x in t:
            x.join()
        assert not bad
    finally:
        for s, _, _ in made:
            s.close()
