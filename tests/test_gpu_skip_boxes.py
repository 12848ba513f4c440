"""Skip boxes and stencil offsets of the raycast at the edges of ragged grids:
scattered single voxels and small solid blocks, some on the grid's faces, so
that rays leave the grid out of boxes that reach beyond it and stencils end at
its last voxel. Both forms of the march (launches of 341, 4800 and 9211 workgroups, on both
sides of the lines between them for 8-byte records) against the instrumented march, which takes every step the
reference takes; the maps are compared bit for bit."""
import numpy as np
import pytest

import vscan

pytestmark = pytest.mark.gpu


def _volume(dims, seed):
    nx, ny, nz = dims
    rng = np.random.default_rng(seed)
    F, W = np.ones((nz, ny, nx), np.float32), np.zeros((nz, ny, nx), np.float32)
    n = max(4, nx * ny * nz // 2000)
    z, y, x = (rng.integers(0, k, n) for k in (nz, ny, nx))
    F[z, y, x], W[z, y, x] = rng.uniform(-1, 1, n).astype(np.float32), 2.0
    for _ in range(12):
        c = [int(rng.integers(0, k)) for k in (nz, ny, nx)]
        s = tuple(slice(max(0, k - 3), k + 4) for k in c)
        F[s] = rng.choice([-1.0, 0.25, -0.25], F[s].shape).astype(np.float32)
        W[s] = 1.0
    return F, W


@pytest.mark.parametrize("dims,tsdf,weight", [
    ((8, 8, 8), vscan.VS_TSDF_F32, vscan.VS_WEIGHT_F32),        # one brick: no stencil reaches a second
    ((40, 24, 16), vscan.VS_TSDF_F16, vscan.VS_WEIGHT_U8),      # superbricks partly outside the grid
    ((264, 200, 312), vscan.VS_TSDF_F32, vscan.VS_WEIGHT_U8),   # odd brick counts
    ((520, 512, 520), vscan.VS_TSDF_F16, vscan.VS_WEIGHT_F32),  # superbricks of 32^3 voxels
])
@pytest.mark.parametrize("w,h", [(321, 243), (1280, 960), (1928, 1208)])
def test_boxes_at_the_edges(ctx, dims, tsdf, weight, w, h):
    print(f"case: {dims} storage {tsdf}/{weight}, {w}x{h}", flush=True)
    st = vscan.SceneStream(3, seed=2, width=w, height=h)
    d = vscan.make_desc(vscan.WORKLOADS["plain_320x240_128"], tsdf=tsdf, weight=weight, K=st.K, W=w, H=h)
    d.voxel = 0.8 / max(dims)
    d.mu = 3 * d.voxel
    for k in range(3):
        d.vol_dim[k] = dims[k]
        d.origin[k] = (-0.5 if k < 2 else -0.2) * dims[k] * d.voxel
    s = vscan.Session(ctx, d, T_gc0=st.pose(0))
    try:
        F, W = _volume(dims, 7)
        s.set_volume(F, W)
        for k in (0, 2):
            s.set_pose(st.pose(k))
            s.raycast(0)
            got = s.maps(0)
            s.raycast_counts(0)
            for a, b in zip(got, s.maps(0)):
                assert np.array_equal(a, b)
            assert (got[0] > 0).any(), "some ray hits"
    finally:
        s.close()
