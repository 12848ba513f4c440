"""Sessions of a batched step closed one after another: the step ran on the
first session's own stream, and the others stay usable (and closable) after
that stream is gone."""
import numpy as np
import pytest

import vscan

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [2, 17])  # one chain, and the parts of a split batch
def test_closing_the_first_session_of_a_batch(ctx, n):
    st = vscan.SceneStream(3, seed=3, width=160, height=120)
    d = vscan.make_desc(vscan.WORKLOADS["plain_320x240_128"], n=64, W=160, H=120, K=st.K)
    sessions = [vscan.Session(ctx, d, T_gc0=st.pose(0)) for _ in range(n)]
    try:
        for k in range(2):
            print(f"case: batch of {n}, step {k}", flush=True)
            ctx.fuse_batch(sessions, [st.frame(k)] * n)
        want = sessions[-1].pose()
        while len(sessions) > 1:
            sessions.pop(0).close()
            for s in sessions:
                assert s.status()[0] == vscan.VS_OK
                assert np.array_equal(s.pose(), want)
    finally:
        for s in sessions:
            s.close()
