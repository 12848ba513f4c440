"""The tracker over sessions of different depth in one batch. In the one-launch
form of the iteration a session with fewer levels than the batch takes part in
some of the launches only, so its pending partials are not always where the
next launch expects them; odd iteration counts shift which half they are in.
Every member is compared bit for bit with the same session fused alone. And
single-level sessions in batches of more than 256 groups (two launches an
iteration) against one alone (one launch)."""
import numpy as np
import pytest

import vscan

pytestmark = pytest.mark.gpu


def session(ctx, st, levels, iters, w, h):
    d = vscan.make_desc(vscan.WORKLOADS["plain_320x240_128"], n=64, W=w, H=h, K=st.K)
    d.levels = levels
    for l in range(3):
        d.iters[l] = iters[l]
    return vscan.Session(ctx, d, T_gc0=st.pose(0))


def groups(w, h):
    tiles = ((w + 31) // 32) * ((h + 7) // 8)
    return (tiles + 7) // 8


@pytest.mark.parametrize("members", [
    [(3, (3, 3, 1)), (1, (4, 0, 0)), (2, (5, 2, 0))],
    [(1, (3, 0, 0)), (2, (2, 1, 0)), (3, (4, 2, 3)), (1, (0, 0, 0))],   # the coarse launches odd in number
    [(2, (10, 5, 0)), (3, (10, 5, 4)), (3, (1, 0, 5)), (3, (2, 3, 0))],  # members that sit out levels
    [(3, (2, 2, 2)), (2, (3, 3, 0)), (1, (9, 0, 0)), (2, (0, 3, 0)), (3, (0, 0, 1))],
])
def test_levels_side_by_side(ctx, members):
    w, h = 320, 240
    print(f"case: one-launch iterations over {members}", flush=True)
    assert len(members) * groups(w, h) <= 256
    st = vscan.SceneStream(3, seed=9, width=w, height=h)
    alone, batch = [], []
    try:
        for levels, iters in members:
            alone.append(session(ctx, st, levels, iters, w, h))
            batch.append(session(ctx, st, levels, iters, w, h))
        solves = 0
        for k in (0, 1, 3, 4):
            mm = st.frame(k)
            ctx.fuse_batch(batch, [mm] * len(batch))
            for a, b, m in zip(alone, batch, members):
                a.fuse(mm)
                assert a.status() == b.status(), (k, m)
                assert np.array_equal(a.pose(), b.pose()), (k, m)
                solves += a.status()[2]
        assert solves > 0
    finally:
        for s in alone + batch:
            s.close()


@pytest.mark.parametrize("w,h,n", [(320, 240, 7), (640, 480, 2)])
@pytest.mark.parametrize("iters", [1, 7])
def test_single_level_in_two_launches(ctx, w, h, n, iters):
    print(f"case: {n} single-level sessions of {w}x{h}, {iters} iterations", flush=True)
    assert groups(w, h) <= 256 < n * groups(w, h) and n < 16  # from 16 sessions a batch runs in parts
    st = vscan.SceneStream(3, seed=9, width=w, height=h)
    made = [session(ctx, st, 1, (iters, 0, 0), w, h) for _ in range(n + 1)]
    lone, many = made[0], made[1:]
    try:
        for k in (0, 1, 3):
            mm = st.frame(k)
            lone.fuse(mm)
            ctx.fuse_batch(many, [mm] * n)
            for s in many:
                assert s.status() == lone.status()
                assert np.array_equal(s.pose(), lone.pose())
        assert lone.status()[2] > 0
    finally:
        for s in made:
            s.close()
