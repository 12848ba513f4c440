"""Both forms of the raycast march in every storage form, address form and ray
block that a launch can take, against the instrumented march, which takes every
step the reference takes; the maps are compared bit for bit.

The ray block comes from a tuning cache, as a context with settled shapes
applies it. The sizes lie on both sides of the lines between the forms: 32768
workgroups for 4-byte records and 8192 for 8-byte ones over grids of small
superbricks, 2048 for larger grids."""
import numpy as np
import pytest

import vscan
from test_gpu_skip_boxes import _volume

pytestmark = pytest.mark.gpu

F32, F16, U8 = vscan.VS_TSDF_F32, vscan.VS_TSDF_F16, vscan.VS_WEIGHT_U8
NAME = {(F32, vscan.VS_WEIGHT_F32): "f32+f32", (F32, U8): "f32+u8", (F16, vscan.VS_WEIGHT_F32): "f16+f32",
        (F16, U8): "f16+u8"}


def groups(w, h):
    return ((w + 31) // 32) * ((h + 7) // 8)


def check(got, s, what):
    s.raycast_counts(0)
    for a, b in zip(got, s.maps(0)):
        assert np.array_equal(a, b), what
    assert (got[0] > 0).any(), "some ray hits"


@pytest.mark.parametrize("block", ["8x8", "16x4", "32x2"])
@pytest.mark.parametrize("dims,tsdf,weight,w,h", [
    ((72, 64, 80), F16, U8, 321, 243),       # latency form, 4-byte records
    ((72, 64, 80), F16, U8, 4096, 2064),     # 33024 workgroups: the wide form, 4-byte records
    ((72, 64, 80), F32, U8, 321, 243),       # latency form, 8-byte records
    ((72, 64, 80), F32, U8, 1928, 1208),     # 9211 workgroups: the wide form, 8-byte records
    ((72, 64, 80), F16, vscan.VS_WEIGHT_F32, 1928, 1208),
    ((72, 64, 80), F32, vscan.VS_WEIGHT_F32, 1928, 1208),
    ((520, 512, 520), F16, U8, 321, 243),    # superbricks of 32^3 voxels: latency form
    ((520, 512, 520), F16, U8, 1280, 960),   # 4800 workgroups: the wide form, superbrick size read per session
])
def test_ray_blocks(dims, tsdf, weight, w, h, block, tmp_path):
    print(f"case: march {block}, {dims} storage {tsdf}/{weight}, {w}x{h}: {groups(w, h)} workgroups", flush=True)
    edge = 1
    while edge < max(dims):
        edge *= 2
    cls = f"{w}x{h} v{edge} {NAME[tsdf, weight]} n1"
    cache = tmp_path / "shapes.txt"
    cache.write_text(f"{cls}|{block}|8x8|2048\n")
    st = vscan.SceneStream(3, seed=2, width=w, height=h)
    d = vscan.make_desc(vscan.WORKLOADS["plain_320x240_128"], tsdf=tsdf, weight=weight, K=st.K, W=w, H=h)
    d.levels = 1
    d.voxel = 0.8 / max(dims)
    d.mu = 3 * d.voxel
    for k in range(3):
        d.vol_dim[k] = dims[k]
        d.origin[k] = (-0.5 if k < 2 else -0.2) * dims[k] * d.voxel
    with vscan.Context(0) as c:
        c.set_tuning(vscan.VS_TUNE_CACHED, str(cache))
        assert c.tuning()[cls]["march"] == block
        s = vscan.Session(c, d, T_gc0=st.pose(0))
        try:
            s.set_volume(*_volume(dims, 7))
            # an empty first frame: nothing to track against, nothing to integrate, the volume is rendered
            s.fuse(np.zeros((h, w), np.uint16))
            check(s.maps(0), s, block)
        finally:
            s.close()


def test_wide_form_over_64_bit_addresses(ctx):
    w, h, dims = 1280, 960, (1024, 1024, 1032)
    print(f"case: wide march of a {dims} grid, {w}x{h}", flush=True)
    assert groups(w, h) > 2048
    st = vscan.SceneStream(3, seed=5, width=w, height=h)
    d = vscan.make_desc(vscan.WORKLOADS["fp16_640x480_512"], K=st.K, W=w, H=h)
    d.levels = 1
    d.voxel = 1.2 / 1024
    d.mu = 3 * d.voxel
    for k in range(3):
        d.vol_dim[k] = dims[k]
        d.origin[k] = (-0.5 if k < 2 else -0.15) * dims[k] * d.voxel
    s = vscan.Session(ctx, d, T_gc0=st.pose(0))
    try:
        for k in range(2):
            s.set_pose(st.pose(k))
            s.set_depth(st.frame(k))
            s.integrate()
        s.raycast(0)
        check(s.maps(0), s, "64-bit")
    finally:
        s.close()
