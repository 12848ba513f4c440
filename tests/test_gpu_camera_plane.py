"""Integration of voxels at, around and behind the camera's own plane, where a
projection divides by a depth of zero or nearly zero: the camera stands inside
the volume, voxel centres lie exactly on its plane (identity pose, a grid of
power-of-two voxels) or a rounding error off it (turned pose), and the surface
is a few millimetres away. Bricks, updated voxels and weights against the
oracle, bit for bit; values within its tolerance of the depth integration."""
import numpy as np
import pytest

import oracle_lib as orc
import vscan

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("turn", [0.0, 0.3])
@pytest.mark.parametrize("depth_mm", [4, 20, 60])
def test_voxels_on_the_camera_plane(ctx, turn, depth_mm):
    print(f"case: surface at {depth_mm} mm, turned by {turn}", flush=True)
    st = vscan.SceneStream(1, seed=1)
    d = vscan.make_desc(vscan.WORKLOADS["plain_320x240_128"], n=64, K=st.K)
    d.voxel = 1.0 / 64
    d.mu = 3.0 / 64
    for k in range(3):
        d.origin[k] = -(31 + 0.5) / 64  # the centre of voxel 31 is 0 on every axis
    T = np.eye(4)
    c, s_ = np.cos(turn), np.sin(turn)
    T[:3, :3] = [[c, 0, s_], [0, 1, 0], [-s_, 0, c]]
    mm = np.full((240, 320), depth_mm, np.uint16)
    mm[::7, ::5] = 0
    s = vscan.Session(ctx, d, T_gc0=T)
    try:
        s.set_pose(T)
        s.set_depth(mm)
        s.integrate()
        F, Wt = np.ones(64 ** 3), np.zeros(64 ** 3)
        Tg, Tc = np.float32(T), np.float32(orc.rigid_inverse(T))
        bm, upd, counts = orc.integrate(mm, orc.K_levels(d)[0], Tg, Tc, orc.volume(d), F, Wt)
        assert s.integrate_counts() == (counts[0], counts[1]) and counts[1] > 0
        gF, gW, _ = s.volume()
        assert np.array_equal(gW.reshape(-1), Wt.astype(np.float32))
        # FP32 SDF of a few mm over mu: two roundings of ~0.06 m and of the
        # quotient, 3 * 2^-24 * 0.06 / mu
        assert np.abs(gF.reshape(-1) - F).max() <= 3 * 2.0 ** -24 * (0.064 + 3 * d.mu) / d.mu + 2.0 ** -23
    finally:
        s.close()
