"""Slot-table sessions fused outside their table, by vs_fuse_batch or as single
sessions: the batched step runs on its first session's own stream, and closing
that session's slot leaves the others usable, with the step's results, whether
or not a server step came in between."""
import numpy as np
import pytest

import vscan

pytestmark = pytest.mark.gpu


def poses(sessions):
    return [s.pose() for s in sessions]


@pytest.mark.parametrize("step_between", [False, True])
@pytest.mark.parametrize("n", [2, 17])  # one chain, and the parts of a split batch
def test_closing_the_first_slot_of_a_batch(ctx, n, step_between):
    print(f"case: {n} slots fused as a batch, closed one after another, server step between: {step_between}", flush=True)
    st = vscan.SceneStream(3, seed=3, width=160, height=120)
    d = vscan.make_desc(vscan.WORKLOADS["plain_320x240_128"], n=64, W=160, H=120, K=st.K)
    server = vscan.Server(ctx, n)
    lone = vscan.Session(ctx, d, T_gc0=st.pose(0))
    try:
        slots = [server.open(d, st.pose(0)) for _ in range(n)]
        for k in range(3):
            ctx.fuse_batch([server.session(i) for i in slots], [st.frame(k)] * n)
            lone.fuse(st.frame(k))
        if step_between:  # the first slot's last stream becomes the server's
            server.step(slots[:1], [st.frame(3)])
        want = lone.pose()
        while len(slots) > 1:
            server.close_slot(slots.pop(0))
            for i in slots:
                s = server.session(i)
                assert s.status()[0] == vscan.VS_OK
                assert np.array_equal(s.pose(), want)
        server.step(slots, [st.frame(4)])
        lone.fuse(st.frame(4))
        assert np.array_equal(server.session(slots[0]).pose(), lone.pose())
    finally:
        lone.close()
        server.close()


def test_single_session_steps_in_a_slot(ctx):
    """A slot closed while its session's own steps are in flight; the memory
    that the next session takes over is written by nothing of the old one."""
    print("case: slots closed behind single-session steps", flush=True)
    st = vscan.SceneStream(3, seed=3, width=320, height=240)
    d = vscan.make_desc(vscan.WORKLOADS["plain_320x240_128"], n=64, W=320, H=240, K=st.K)
    server = vscan.Server(ctx, 2)
    lone = vscan.Session(ctx, d, T_gc0=st.pose(0))
    try:
        lone.fuse(st.frame(0))
        want, vol = lone.pose(), lone.volume()
        for _ in range(4):
            a = server.open(d, st.pose(0))
            for k in range(4):
                server.session(a).fuse(st.frame(k))
            server.close_slot(a)
            b = server.open(d, st.pose(0))
            server.step([b], [st.frame(0)])
            s = server.session(b)
            assert s.status()[:2] == (vscan.VS_OK, 1)
            assert np.array_equal(s.pose(), want)
            for x, y in zip(s.volume(), vol):
                assert np.array_equal(x, y)
            server.close_slot(b)
    finally:
        lone.close()
        server.close()
