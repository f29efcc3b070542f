"""Stage entry points called out of order are refused on the host with MSPLAT_ERR_ARG,
before any kernel launch: a raster or loss stage with no binned frame, a backward with no
render, and any of them after msplat_hip_radix_sort ended the frame. Each
refusal leaves the context usable: a full render afterwards still matches a fresh one.
"""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

ERR_ARG = 1
BG = np.array([0.613, 0.0101, 0.3984], np.float32)


def _scene():
    from msplat.camera import look_at, make_camera
    from msplat.scenes import random_scene
    sc = random_scene(3, 500, degree=1, log_scale=(-3.5, 0.5))
    cam = make_camera(look_at((2.5, 0.7, 2.9), (0.1, -0.2, 0)), 64, 48, 60.0, 60.0, dtu=1)
    return sc, cam


def test_out_of_order_stages_are_refused():
    from msplat._abi import Context, DeviceArray, Grads, check, floats, lib, make_camera_struct
    from msplat.backend import DeviceGaussians, render_numpy
    sc, cam = _scene()
    ctx = Context(0)
    try:
        dg = DeviceGaussians(ctx, sc)
        g, c = dg.struct(), make_camera_struct(cam, 1)
        L = lib()
        gt = DeviceArray(ctx, (cam["H"], cam["W"], 3))
        v_img = DeviceArray(ctx, (cam["H"], cam["W"], 3))
        out = {k: DeviceArray(ctx, (dg.n, dg.widths[k])) for k in ("means", "scales", "quats", "dc", "rest", "opac")}
        gr = Grads(*[out[k].ptr for k in ("means", "scales", "quats", "dc", "rest", "opac")])
        loss = C.c_float()
        # a fresh context holds no frame
        assert L.msplat_hip_stage_bin(ctx.ptr, C.byref(c)) == ERR_ARG
        assert L.msplat_hip_stage_raster_forward(ctx.ptr, C.byref(c), floats(BG)) == ERR_ARG
        assert L.msplat_hip_stage_loss(ctx.ptr, C.byref(c), C.c_void_p(gt.ptr), 0.2, 1e-3, C.byref(loss)) == ERR_ARG
        assert L.msplat_hip_render_backward(ctx.ptr, C.byref(g), C.byref(c), floats(BG), C.c_void_p(v_img.ptr),
                                            C.byref(gr)) == ERR_ARG
        # projected but not binned
        check(L.msplat_hip_stage_project(ctx.ptr, C.byref(g), C.byref(c)))
        assert L.msplat_hip_stage_raster_forward(ctx.ptr, C.byref(c), floats(BG)) == ERR_ARG
        assert L.msplat_hip_render_backward(ctx.ptr, C.byref(g), C.byref(c), floats(BG), C.c_void_p(v_img.ptr),
                                            C.byref(gr)) == ERR_ARG
        # binned, not rasterized: the loss and the backward still need an image
        check(L.msplat_hip_stage_bin(ctx.ptr, C.byref(c)))
        assert L.msplat_hip_stage_loss(ctx.ptr, C.byref(c), C.c_void_p(gt.ptr), 0.2, 1e-3, C.byref(loss)) == ERR_ARG
        # a rendered frame, then a radix sort, which ends it
        ref = render_numpy(ctx, dg, cam, BG)
        keys = DeviceArray.from_numpy(ctx, np.arange(100, 0, -1, dtype=np.uint64))
        vals = DeviceArray.from_numpy(ctx, np.arange(100, dtype=np.int32))
        check(L.msplat_hip_radix_sort(ctx.ptr, C.c_void_p(keys.ptr), C.c_void_p(vals.ptr), 100, 32))
        assert L.msplat_hip_stage_raster_forward(ctx.ptr, C.byref(c), floats(BG)) == ERR_ARG
        assert L.msplat_hip_render_backward(ctx.ptr, C.byref(g), C.byref(c), floats(BG), C.c_void_p(v_img.ptr),
                                            C.byref(gr)) == ERR_ARG
        assert L.msplat_hip_stage_loss(ctx.ptr, C.byref(c), C.c_void_p(gt.ptr), 0.2, 1e-3, C.byref(loss)) == ERR_ARG
        np.testing.assert_array_equal(keys.numpy(), np.arange(1, 101, dtype=np.uint64))
        # re-binning the still-projected frame makes it usable again
        check(L.msplat_hip_stage_bin(ctx.ptr, C.byref(c)))
        check(L.msplat_hip_stage_raster_forward(ctx.ptr, C.byref(c), floats(BG)))
        img = ctx.download(ctx.frame().image, (cam["H"], cam["W"], 3), np.float32)
        np.testing.assert_array_equal(img, ref)
        np.testing.assert_array_equal(render_numpy(ctx, dg, cam, BG), ref)
        ctx.sync()
    finally:
        ctx.close()


def test_lists_are_offered_for_a_binned_frame_only():
    """A frame that is projected, or whose radix sort ended it, has no lists: the earlier
    frame's ids and ranges are not offered, nor read for the 64-bit keys of the new one's
    tiles. Binned, they are the new frame's."""
    from msplat._abi import FRAME_KEYS64, Context, DeviceArray, check, lib, make_camera_struct
    from msplat.backend import DeviceGaussians, render_numpy
    from msplat.camera import look_at, make_camera
    sc, small = _scene()
    large = make_camera(look_at((2.5, 0.7, 2.9), (0.1, -0.2, 0)), 320, 240, 300.0, 300.0, dtu=1)
    ctx = Context(0)
    try:
        dg, L = DeviceGaussians(ctx, sc), lib()
        ctx.set_flags(FRAME_KEYS64)
        render_numpy(ctx, dg, small, BG)
        assert ctx.frame().isect_gid and ctx.frame().isect_keys
        g, c = dg.struct(), make_camera_struct(large, 1)
        check(L.msplat_hip_stage_project(ctx.ptr, C.byref(g), C.byref(c)))
        f = ctx.frame()
        assert f.num_tiles == 20 * 15 and not f.isect_gid and not f.isect_keys
        check(L.msplat_hip_stage_bin(ctx.ptr, C.byref(c)))
        f = ctx.frame()
        M = int(f.num_isects)
        start = ctx.download(f.tile_start, (f.num_tiles + 1,), np.int32)
        keys = ctx.download(f.isect_keys, (M,), np.uint64)
        assert start[-1] == M > 0
        np.testing.assert_array_equal(keys >> np.uint64(32), np.repeat(np.arange(f.num_tiles), np.diff(start)))
        depths = ctx.download(f.depths, (dg.n,), np.float32)
        np.testing.assert_array_equal((keys & np.uint64(0xFFFFFFFF)).astype(np.uint32),
                                      depths[ctx.download(f.isect_gid, (M,), np.int32)].view(np.uint32))
        sorted_keys = DeviceArray.from_numpy(ctx, np.arange(100, 0, -1, dtype=np.uint64))
        vals = DeviceArray.from_numpy(ctx, np.arange(100, dtype=np.int32))
        check(L.msplat_hip_radix_sort(ctx.ptr, C.c_void_p(sorted_keys.ptr), C.c_void_p(vals.ptr), 100, 32))
        f = ctx.frame()
        assert not f.isect_gid and not f.isect_keys
    finally:
        ctx.close()


def test_a_sort_before_the_first_frame():
    """A radix sort as a context's first call leaves the running counts of its frames zero and
    all of them allocated (it needs only the element count among those scalars)."""
    from msplat._abi import Context, DeviceArray, check, lib
    from msplat.backend import DeviceGaussians, render_numpy
    sc, cam = _scene()
    ctx = Context(0)
    try:
        keys = DeviceArray.from_numpy(ctx, np.arange(100, 0, -1, dtype=np.uint64))
        vals = DeviceArray.from_numpy(ctx, np.arange(100, dtype=np.int32))
        check(lib().msplat_hip_radix_sort(ctx.ptr, C.c_void_p(keys.ptr), C.c_void_p(vals.ptr), 100, 32))
        np.testing.assert_array_equal(vals.numpy(), np.arange(99, -1, -1, dtype=np.int32))
        dg = DeviceGaussians(ctx, sc)
        for frames in range(3):
            f = ctx.frame()
            assert ctx.download(f.isects_running, (1,), np.uint64)[0] == frames * f.num_isects
            assert ctx.download(f.visible_running, (1,), np.uint64)[0] == frames * f.num_visible
            assert ctx.download(f.slots_written, (1,), np.uint64)[0] == 0
            render_numpy(ctx, dg, cam, BG)
        assert ctx.frame().num_isects > 0
    finally:
        ctx.close()
