"""Restored sessions continue bit for bit in every storage form, with colour,
and with every remainder of the stored brick count (the bricks follow the
index list in one upload and have to stay aligned); reset after use gives a
session that fuses like a new one."""
import numpy as np
import pytest

import vscan

pytestmark = pytest.mark.gpu
W0 = vscan.WORKLOADS["plain_320x240_128"]
FORMS = [(vscan.VS_TSDF_F32, vscan.VS_WEIGHT_F32, False), (vscan.VS_TSDF_F32, vscan.VS_WEIGHT_U8, True),
         (vscan.VS_TSDF_F16, vscan.VS_WEIGHT_F32, False), (vscan.VS_TSDF_F16, vscan.VS_WEIGHT_U8, True)]


def desc(st, tsdf, weight, color, n=64):
    mode = vscan.VS_INTEGRATE_COLOR if color else vscan.VS_INTEGRATE_DEPTH
    return vscan.make_desc(W0, tsdf=tsdf, weight=weight, n=n, W=st.W, H=st.H, K=st.K, integrate_mode=mode)


def fuse(s, st, k, color):
    if color:
        y, x = np.mgrid[0:st.H, 0:st.W]
        s.set_color(np.stack([40 + (x + k) % 200, 40 + (y + k) % 200, 40 + (x + y) % 200]).astype(np.uint8))
    s.fuse(st.frame(k))


def same(a, b, color):
    assert np.array_equal(a.pose(), b.pose()) and a.status() == b.status()
    (Fa, Wa, ma), (Fb, Wb, mb) = a.volume(), b.volume()
    assert np.array_equal(Fa, Fb) and np.array_equal(Wa, Wb)
    if a.status()[0] == vscan.VS_OK:  # a frame that was not fused leaves the last mask, which snapshots do not hold
        assert np.array_equal(ma, mb)
    for l in range(3):
        for x, y in zip(a.maps(l), b.maps(l)):
            assert np.array_equal(x, y)
        if color:
            assert np.array_equal(a.texture(l), b.texture(l))
    if color:
        assert np.array_equal(a.volume_color(), b.volume_color())


@pytest.mark.parametrize("tsdf,weight,color", FORMS)
def test_restore_continues(ctx, tsdf, weight, color):
    seen = set()
    for seed in range(1, 25):
        st = vscan.SceneStream(3, seed=seed, width=160, height=120)
        s = vscan.Session(ctx, desc(st, tsdf, weight, color), T_gc0=st.pose(0))
        try:
            fuse(s, st, 0, color)
            data = s.snapshot()
            rest = vscan.SnapshotHeader.from_buffer_copy(data[:500] + bytes(500)).bricks_stored % 4
            if rest in seen:
                continue
            seen.add(rest)
            print(f"case: restore, forms {tsdf} {weight} colour {color}, stored bricks % 4 = {rest}", flush=True)
            r = vscan.restore(ctx, data)
            try:
                for k in (1, 2):
                    fuse(s, st, k, color)
                    fuse(r, st, k, color)
                    same(s, r, color)
            finally:
                r.close()
        finally:
            s.close()
        if len(seen) == 4:
            break
    assert len(seen) >= 3


@pytest.mark.parametrize("tsdf,weight,color", FORMS[:2])
def test_reset_is_a_new_session(ctx, tsdf, weight, color):
    st = vscan.SceneStream(3, seed=7, width=160, height=120)
    d = desc(st, tsdf, weight, color, n=72)  # 729 bricks: not a multiple of 32 or 128
    used = vscan.Session(ctx, d, T_gc0=st.pose(9))
    fresh = vscan.Session(ctx, d, T_gc0=st.pose(0))
    try:
        for k in (9, 10, 11):
            fuse(used, st, k, color)
        T = np.ascontiguousarray(st.pose(0)).reshape(16)
        vscan.check(vscan.lib().vs_session_reset(used.h, vscan._ptr(T), None), "vs_session_reset")
        for k in (0, 1, 2):
            fuse(used, st, k, color)
            fuse(fresh, st, k, color)
        same(used, fresh, color)
    finally:
        used.close()
        fresh.close()
