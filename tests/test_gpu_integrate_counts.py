"""vs_get_integrate_counts reports the last integration until the next one: a
track or a raycast in between, called operator by operator, leaves the counts
as they are, in both forms of the iteration; an integration or a fused step
sets them anew."""
import pytest

import vscan

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("w,h", [(320, 240), (1280, 960)])  # 38 and 600 level-0 groups: one and two launches an iteration
def test_counts_outlive_a_track(ctx, w, h):
    print(f"case: integrate, track, counts at {w}x{h}", flush=True)
    st = vscan.SceneStream(4, seed=1, width=w, height=h)
    d = vscan.make_desc(vscan.WORKLOADS["plain_320x240_128"], W=w, H=h, K=st.K)
    s = vscan.Session(ctx, d, T_gc0=st.pose(0))
    try:
        s.fuse(st.frame(0))
        fused = s.integrate_counts()
        assert fused[0] > 0 and fused[1] > 0
        s.set_depth(st.frame(1))
        s.integrate()
        first = s.integrate_counts()
        assert first[0] > 0 and first[1] > 0
        s.bilateral()
        s.pyramid()
        s.track()
        assert s.status()[0] == vscan.VS_OK
        assert s.integrate_counts() == first
        s.raycast(0)
        s.track()
        assert s.integrate_counts() == first
        s.integrate()
        second = s.integrate_counts()
        s.integrate()
        assert s.integrate_counts() == second, "each integration counts from zero"
        s.fuse(st.frame(2))
        after = s.integrate_counts()
        assert 0 < after[0] < second[0] + first[0] and after[1] > 0
    finally:
        s.close()


def test_counts_of_a_refused_frame(ctx):
    """A fused step whose track is refused integrates nothing."""
    print("case: counts of a refused frame", flush=True)
    st = vscan.SceneStream(4, seed=1, width=320, height=240)
    d = vscan.make_desc(vscan.WORKLOADS["plain_320x240_128"], W=320, H=240, K=st.K)
    d.max_motion_m = 1e-7
    s = vscan.Session(ctx, d, T_gc0=st.pose(0))
    try:
        s.fuse(st.frame(0))
        assert s.integrate_counts()[0] > 0
        s.fuse(st.frame(3))
        assert s.status()[0] == vscan.VS_MOTION_REJECTED
        assert s.integrate_counts() == (0, 0)
    finally:
        s.close()
