"""The one-launch and the two-launch Gauss-Newton iterations give the same
bits: a session tracked alone (one launch per iteration up to 256 level-0
groups) against copies of it in a batch of more groups (two launches)."""
import numpy as np
import pytest

import vscan

pytestmark = pytest.mark.gpu


def run(ctx, d, st, n, frames):
    sessions = [vscan.Session(ctx, d, T_gc0=st.pose(0)) for _ in range(n)]
    try:
        out = []
        for k in frames:
            mm = st.frame(k)
            ctx.fuse_batch(sessions, [mm] * n)
            out.append([(s.status(), s.pose()) for s in sessions])
        return out
    finally:
        for s in sessions:
            s.close()


@pytest.mark.parametrize("w,h,levels,iters,gate", [
    (320, 240, 3, (10, 5, 4), {}),             # 38 groups, a remainder of 4 tiles
    (333, 251, 2, (3, 2, 0), {}),              # odd tiles, no coarsest level
    (160, 130, 1, (7, 0, 0), {}),              # one level
    (640, 480, 3, (10, 5, 4), {}),             # 150 groups
    (832, 624, 3, (2, 1, 1), {}),              # 254 groups: the last size with one launch below 256
    (320, 240, 3, (0, 0, 0), {}),              # no iteration at all
    (320, 240, 3, (10, 5, 4), {"icp_min_valid": 10 ** 7}),   # every solve refused: too few points
    (320, 240, 3, (10, 5, 4), {"icp_rel_pivot": 0.9}),       # refused as singular
    (320, 240, 3, (10, 5, 4), {"max_motion_m": 1e-7}),       # solved, then gated
])
def test_forms_agree(ctx, w, h, levels, iters, gate):
    print(f"case: {w}x{h} levels {levels} iterations {iters} {gate}", flush=True)
    st = vscan.SceneStream(3, seed=9, width=w, height=h)
    d = vscan.make_desc(vscan.WORKLOADS["plain_320x240_128"], n=64, W=w, H=h, K=st.K)
    d.levels = levels
    for l in range(3):
        d.iters[l] = iters[l]
    for k, v in gate.items():
        setattr(d, k, v)
    tiles = ((w + 31) // 32) * ((h + 7) // 8)
    groups = (tiles + 7) // 8
    lone = run(ctx, d, st, 1, (0, 1, 3))
    many = run(ctx, d, st, min(15, 256 // groups + 1), (0, 1, 3))
    for a, b in zip(lone, many):
        for got in b:
            assert got[0] == a[0][0]
            assert np.array_equal(got[1], a[0][1])
    status, fused, solves = lone[1][0][0]
    if not gate and sum(iters):
        assert status == vscan.VS_OK and solves > 0
    if "icp_min_valid" in gate:
        assert status == vscan.VS_TOO_FEW_POINTS and solves == 1
    if "icp_rel_pivot" in gate:
        assert status == vscan.VS_SINGULAR and solves == 1
    if "max_motion_m" in gate:
        assert status == vscan.VS_MOTION_REJECTED
