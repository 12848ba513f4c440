"""A small download does not wait for a large one of the same context to end:
only the staging lanes, which it does not use, are taken in turn."""
import threading
import time

import numpy as np
import pytest

import vscan

pytestmark = pytest.mark.gpu


def test_small_beside_large(ctx):
    print("case: a 32^3 volume downloaded while a 512^3 one is", flush=True)
    w = vscan.WORKLOADS["fp16_640x480_512"]
    big = vscan.Session(ctx, vscan.make_desc(w, n=512, W=64, H=48, K=(60.0, 60.0, 31.5, 23.5)))
    small = vscan.Session(ctx, vscan.make_desc(w, n=32, W=64, H=48, K=(60.0, 60.0, 31.5, 23.5)))
    F, W, f = np.ones(512 ** 3, np.float32), np.ones(512 ** 3, np.float32), np.zeros(32 ** 3, np.float32)
    shares = []
    try:
        def download(s, *to):
            vscan.check(vscan.lib().vs_volume_download(s.h, *[vscan._ptr(a) for a in to], None), "vs_volume_download")

        download(big, F, W)
        for _ in range(3):
            span = []

            def work():
                t = time.perf_counter()
                download(big, F, W)
                span.append(time.perf_counter() - t)

            t = threading.Thread(target=work)
            t.start()
            longest = 0.0
            while t.is_alive():
                t0 = time.perf_counter()
                download(small, f, None)
                longest = max(longest, time.perf_counter() - t0)
            t.join()
            shares.append(longest / span[0])
        print("longest small download, as shares of the large one's time:", shares, flush=True)
        assert (f == 1.0).all()
        # 0.03-0.05 where it waits for single copies, 0.95-0.98 where it waits for the large one's end
        assert min(shares) < 0.5
    finally:
        big.close()
        small.close()
