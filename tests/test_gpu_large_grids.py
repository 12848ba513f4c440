"""Raycast of grids around the size where a superbrick of 16^3 voxels no longer
fits the distance field's LDS copy (32768 cells): the march with its skips
against the instrumented march, which takes every step the reference takes.
The maps are compared bit for bit."""
import numpy as np
import pytest

import vscan

pytestmark = pytest.mark.gpu

CASES = [
    ((512, 512, 512), vscan.VS_TSDF_F16, vscan.VS_WEIGHT_U8),   # 32^3 cells: the last grid with 16^3 voxels a cell
    ((520, 512, 520), vscan.VS_TSDF_F16, vscan.VS_WEIGHT_U8),   # 33 x 32 x 33: 32^3 voxels a cell
    ((1024, 504, 168), vscan.VS_TSDF_F32, vscan.VS_WEIGHT_U8),  # 64 x 32 x 11 cells of 16^3: the last that fits
    ((2048, 512, 136), vscan.VS_TSDF_F32, vscan.VS_WEIGHT_F32),  # flat and wide, partial cells along z
    ((1024, 1024, 1032), vscan.VS_TSDF_F16, vscan.VS_WEIGHT_U8),  # records above 4 GB, 64^3 voxels a cell
]


@pytest.mark.parametrize("dims,tsdf,weight", CASES)
def test_skips_change_no_ray(ctx, dims, tsdf, weight):
    print(f"case: raycast of a {dims} grid", flush=True)
    st = vscan.SceneStream(3, seed=5, width=320, height=240)
    d = vscan.make_desc(vscan.WORKLOADS["fp16_640x480_512"], tsdf=tsdf, weight=weight, K=st.K, W=320, H=240)
    d.voxel = 1.2 / min(max(dims), 1024)
    d.mu = 3 * d.voxel
    for k in range(3):
        d.vol_dim[k] = dims[k]
        d.origin[k] = (-0.5 if k < 2 else -0.15) * dims[k] * d.voxel
    s = vscan.Session(ctx, d, T_gc0=st.pose(0))
    try:
        for k in range(3):
            s.set_pose(st.pose(k))
            s.set_depth(st.frame(k))
            s.integrate()
        for l in range(3):
            s.raycast(l)
            got = s.maps(l)
            s.raycast_counts(l)
            ref = s.maps(l)
            assert (got[0] > 0).sum() > 0.2 * got[0].size, "the scene fills a part of the frame"
            for a, b in zip(got, ref):
                assert np.array_equal(a, b)
    finally:
        s.close()
