"""Pose, status and frame count as the host reads them: after every call that
changes them, across reset and restore, and for a slot whose session is closed
while steps are in flight and whose record is then taken by a new session."""
import numpy as np
import pytest

import vscan

pytestmark = pytest.mark.gpu
W0 = vscan.WORKLOADS["plain_320x240_128"]


def desc(st, n=64):
    return vscan.make_desc(W0, tsdf=vscan.VS_TSDF_F16, weight=vscan.VS_WEIGHT_U8, n=n, W=st.W, H=st.H, K=st.K)


def test_after_every_change(ctx):
    st = vscan.SceneStream(3, seed=3, width=160, height=120)
    s = vscan.Session(ctx, desc(st), T_gc0=st.pose(0))
    try:
        assert np.array_equal(s.pose(), st.pose(0)) and s.status() == (0, 0, 0)
        s.fuse(st.frame(0))
        assert s.status() == (0, 1, 0)
        s.fuse(st.frame(1))
        status, frames, solves = s.status()
        assert (status, frames) == (0, 2) and solves > 0
        tracked = s.pose()
        assert not np.array_equal(tracked, st.pose(0))
        data = s.snapshot()
        hdr = vscan.SnapshotHeader.from_buffer_copy(data[:500] + bytes(500))
        assert np.array_equal(np.array(hdr.T_gc).reshape(4, 4), tracked) and hdr.frames == 2
        r = vscan.restore(ctx, data)
        try:
            assert np.array_equal(r.pose(), tracked) and r.status()[1] == 2
        finally:
            r.close()
        s.set_pose(st.pose(5))
        assert np.array_equal(s.pose(), st.pose(5)) and s.status()[1] == 2
        T = np.ascontiguousarray(st.pose(7)).reshape(16)
        vscan.check(vscan.lib().vs_session_reset(s.h, vscan._ptr(T), None), "vs_session_reset")
        assert np.array_equal(s.pose(), st.pose(7)) and s.status() == (0, 0, 0)
    finally:
        s.close()


def test_reopened_slots_keep_their_own(ctx):
    st = vscan.SceneStream(3, seed=4, width=160, height=120)
    srv = vscan.Server(ctx, 4, vscan.VS_TSDF_F16, vscan.VS_WEIGHT_U8)
    try:
        for rnd in range(20):
            slots = [srv.open(desc(st), T_gc0=st.pose(k + rnd)) for k in range(4)]
            for k in range(3):
                srv.step(slots, [st.frame(k)] * 4)  # in flight when the slots close
            for i in slots:
                srv.close_slot(i)
            fresh = [srv.open(desc(st), T_gc0=st.pose(20 + k)) for k in range(4)]
            for k, i in enumerate(fresh):
                assert np.array_equal(srv.session(i).pose(), st.pose(20 + k))
                assert srv.session(i).status() == (0, 0, 0)
            for i in fresh:
                srv.close_slot(i)
    finally:
        srv.close()
