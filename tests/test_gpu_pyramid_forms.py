"""Pyramid levels 1 and 2 in one launch on both sides of 768 level-2 tiles, above
which a tile takes 4 waves instead of 16, against the oracle."""
import numpy as np
import pytest

import oracle_lib as orc
import vscan

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("w,h,tiles", [(2051, 1537, 768), (2053, 1540, 833), (2603, 2001, 1323)])
def test_tile_counts(ctx, w, h, tiles):
    w2, h2 = w >> 2, h >> 2
    n = ((w2 + 31) // 32) * ((h2 + 7) // 8)
    print(f"case: pyramid of {w}x{h}, {n} level-2 tiles", flush=True)
    assert n == tiles
    rng = np.random.default_rng(w)
    img = rng.uniform(0.5, 3.0, (h, w)).astype(np.float32)
    img[rng.random((h, w)) < 0.1] = 0
    d = vscan.make_desc(vscan.WORKLOADS["plain_320x240_128"], n=16, W=w, H=h, K=(w * 0.8, w * 0.8, w / 2, h / 2))
    s = vscan.Session(ctx, d)
    try:
        s.set_filtered(0, img)
        s.pyramid()
        s.sync()
        for l in (1, 2):
            got = s.filtered(l)
            want = orc.pyr_down(s.filtered(l - 1))
            # three products of at most 6 x 3.0 a row, five rows: under 32 roundings of values below 48, over 256
            assert np.abs(got - want).max() <= 32 * 48 * 2.0 ** -24 / 256 * 16
            assert np.array_equal(got == 0, want == 0)
    finally:
        s.close()
