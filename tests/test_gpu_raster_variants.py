"""The rasterizers' branches: batches with and without opacities at the alpha clamp (0.999),
batches where pixels terminate, tiles of one record and of several batches, every pixels
per lane and batch depth; the images, final T and last indices against the oracle's, the
gradients against the oracle's. Bars are the ones the parity tests use for the same
quantities (1e-5 and 1e-4 relative L2): the two sides round exp and the sums differently."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

BG = np.array([0.613, 0.0101, 0.3984], np.float32)


def _rel(a, b):
    return float(np.linalg.norm(np.asarray(a, np.float64) - b) / max(np.linalg.norm(np.asarray(b, np.float64)), 1e-30))


@pytest.mark.parametrize("ppt,bb,fb", [(4, 64, 256), (4, 32, 64), (2, 128, 128), (1, 64, 256)])
@pytest.mark.parametrize("n,opac,scale", [
    (2500, (9.0, 1.0), -3.0),   # nearly every opacity at the clamp: pixels end after a few records
    (2500, (4.0, 4.0), -3.2),   # batches of both kinds
    (2500, (-3.0, 1.0), -2.2),  # faint and large: long lists, no pixel ends
    (1, (12.0, 0.0), -1.5),     # one clamped record over several tiles
])
def test_rasterizers_match_oracle(oracle, ppt, bb, fb, n, opac, scale):
    from msplat._abi import (FRAME_KEEP_GRADS, TUNE_BWD_BATCH, TUNE_BWD_PPT, TUNE_CHUNKS, TUNE_FWD_BATCH, Context,
                             DeviceArray)
    from msplat.backend import DeviceGaussians, render, render_backward
    from msplat.camera import look_at, make_camera
    from msplat.scenes import random_scene
    W, H = 117, 75
    sc = random_scene(71, n, degree=0, log_scale=(scale, 0.5), opac=opac)
    if n == 1:
        sc["means"][:] = 0.1
    cam = make_camera(look_at((2.2, 0.4, 2.6), (0, 0, 0)), W, H, 110.0, 104.0)
    ctx = Context(0)
    for key, v in ((TUNE_BWD_PPT, ppt), (TUNE_BWD_BATCH, bb), (TUNE_FWD_BATCH, fb), (TUNE_CHUNKS, 1)):
        ctx.set_tuning(key, v)
    ctx.set_flags(FRAME_KEEP_GRADS)
    dg = DeviceGaussians(ctx, sc)
    img = ctx.download(render(ctx, dg, cam, BG), (H, W, 3), np.float32)
    p, b, fwd = oracle.render(sc, cam, BG)
    assert _rel(img, fwd["img"]) < 1e-5
    f = ctx.frame()
    last = ctx.download(f.final_idx, (H, W), np.int32)
    # a pair on a cut-off may fall on its other side
    assert np.mean(last == fwd["final_idx"].reshape(H, W)) > 0.998
    v_img = (np.random.default_rng(9).normal(0, 1, (H, W, 3)) * 1e-3).astype(np.float32)
    render_backward(ctx, dg, cam, BG, DeviceArray.from_numpy(ctx, v_img))
    f = ctx.frame()
    red = oracle.reduce_slots(n, b, oracle.raster_backward(b, fwd, cam, BG, v_img))
    for k, ptr, shape in (("v_xy", f.v_xy, (n, 2)), ("v_conic", f.v_conic, (n, 3)), ("v_rgb", f.v_rgb, (n, 3)),
                          ("v_opac", f.v_opacity, (n,))):
        assert _rel(ctx.download(ptr, shape, np.float32), red[k].reshape(shape)) < 1e-4, k
    ctx.close()


def test_a_pixel_without_a_finite_gradient_spares_what_it_does_not_see():
    """An infinite and a NaN upstream gradient reach the records that the pixel composites;
    the positions and conics of the others (also those in the pixel's tile) stay finite."""
    from msplat._abi import FRAME_KEEP_GRADS, TUNE_CHUNKS, Context, DeviceArray
    from msplat.backend import DeviceGaussians, render, render_backward
    from msplat.camera import look_at, make_camera
    from msplat.scenes import random_scene
    W = H = 32
    sc = random_scene(3, 400, degree=0, log_scale=(-3.6, 0.2), opac=(0.0, 1.0))
    cam = make_camera(look_at((0, 0, 4), (0, 0, 0)), W, H, 60.0, 60.0)
    ctx = Context(0)
    ctx.set_tuning(TUNE_CHUNKS, 1)
    ctx.set_flags(FRAME_KEEP_GRADS)
    dg = DeviceGaussians(ctx, sc)
    render(ctx, dg, cam, BG)
    f = ctx.frame()
    A = ctx.download(f.splat_a, (400, 4), np.float32)
    for bad in (np.inf, np.nan):
        v = np.full((H, W, 3), 1e-3, np.float32)
        v[5, 5] = bad
        render_backward(ctx, dg, cam, BG, DeviceArray.from_numpy(ctx, v))
        f = ctx.frame()
        g = np.concatenate([ctx.download(f.v_xy, (400, 2), np.float32), ctx.download(f.v_conic, (400, 3), np.float32)], 1)
        far = np.hypot(A[:, 0] - 5, A[:, 1] - 5) > 9.0  # beyond any splat's reach (sigma < 2.2 px)
        assert far.sum() > 200 and np.isfinite(g[far]).all()
        assert not np.isfinite(g[~far]).all()
    ctx.close()


@pytest.mark.parametrize("chunks", [1, 3])
def test_an_opacity_that_is_not_a_number(oracle, chunks):
    """min(0.999, NaN) is 0.999, in the reference and here: such a record composites as an
    opaque one, and every gradient but its own opacity's is finite."""
    from msplat._abi import FRAME_KEEP_GRADS, TUNE_CHUNKS, Context, DeviceArray
    from msplat.backend import DeviceGaussians, render, render_backward
    from msplat.camera import look_at, make_camera
    from msplat.scenes import random_scene
    n, W, H = 600, 97, 71
    sc = random_scene(23, n, degree=0, log_scale=(-3.4, 0.3), opac=(-1.0, 1.0))
    sc["opac"][::15] = np.nan
    cam = make_camera(look_at((2.2, 0.4, 2.6), (0, 0, 0)), W, H, 90.0, 88.0)
    ctx = Context(0)
    ctx.set_tuning(TUNE_CHUNKS, chunks)
    ctx.set_flags(FRAME_KEEP_GRADS)
    dg = DeviceGaussians(ctx, sc)
    img = ctx.download(render(ctx, dg, cam, BG), (H, W, 3), np.float32)
    p, b, fwd = oracle.render(sc, cam, BG)
    assert _rel(img, fwd["img"]) < 1e-5
    f = ctx.frame()
    last = ctx.download(f.final_idx, (H, W), np.int32)
    assert np.mean(last == fwd["final_idx"].reshape(H, W)) > 0.998
    v_img = (np.random.default_rng(9).normal(0, 1, (H, W, 3)) * 1e-3).astype(np.float32)
    render_backward(ctx, dg, cam, BG, DeviceArray.from_numpy(ctx, v_img))
    f = ctx.frame()
    red = oracle.reduce_slots(n, b, oracle.raster_backward(b, fwd, cam, BG, v_img))
    number = np.isfinite(sc["opac"][:, 0])
    for k, ptr, shape in (("v_xy", f.v_xy, (n, 2)), ("v_conic", f.v_conic, (n, 3)), ("v_rgb", f.v_rgb, (n, 3)),
                          ("v_opac", f.v_opacity, (n,))):
        got, want = ctx.download(ptr, shape, np.float32), red[k].reshape(shape)
        if k == "v_opac":
            got, want = got[number], want[number]
        assert np.isfinite(got).all() and _rel(got, want) < 1e-4, k
    ctx.close()
