"""Pyramid levels 1 and 2 in one launch at the edges of its tiles: level-1
sizes that are odd, one tile, or exactly whole tiles of 64x16 (whose odd last
column or row the last tile owns), against the oracle; and the same levels
when a two-level session in the batch keeps the launches apart."""
import numpy as np
import pytest

import oracle_lib as orc
import vscan

pytestmark = pytest.mark.gpu
W0 = vscan.WORKLOADS["plain_320x240_128"]


def session(ctx, w, h, levels):
    d = vscan.make_desc(W0, n=16, W=w, H=h, K=(w * 0.8, w * 0.8, w / 2, h / 2))
    d.levels = levels
    return vscan.Session(ctx, d)


@pytest.mark.parametrize("w,h", [(16, 16), (17, 19), (128, 32), (130, 34), (131, 35), (258, 66), (259, 67), (333, 251),
                                 (640, 480), (643, 481)])
def test_levels(ctx, w, h):
    print(f"case: pyramid of {w}x{h}", flush=True)
    rng = np.random.default_rng(w + h)
    img = rng.uniform(0.5, 3.0, (h, w)).astype(np.float32)
    img[rng.random((h, w)) < 0.1] = 0
    s = session(ctx, w, h, 3)
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


def test_two_levels_beside_three(ctx):
    print("case: batch of a two-level and a three-level session", flush=True)
    st = vscan.SceneStream(3, seed=2, width=259, height=131)
    sessions = [session(ctx, 259, 131, n) for n in (2, 3, 3)]
    lone = session(ctx, 259, 131, 3)
    try:
        mm = st.frame(0)
        ctx.fuse_batch(sessions, [mm] * 3)
        lone.fuse(mm)
        for l in range(3):
            want = lone.filtered(l)
            for s in sessions:
                if l < s.desc.levels:
                    assert np.array_equal(s.filtered(l), want)
    finally:
        for s in sessions + [lone]:
            s.close()
