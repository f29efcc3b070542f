"""The tiles' lists (tile_lists.hip) against a host restatement from the frame's own
projection outputs: every tile's gaussians ascending by (depth bits, id), at the edges of
the two expansion levels (8 tiles, 64 tiles), of the 64-entry groups, and with splats from
under a tile to the whole view. Whole numbers: exact."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

BG = np.array([0.613, 0.0101, 0.3984], np.float32)


def _expected(ctx, f, n, tiles_x, tiles_y):
    xy = ctx.download(f.splat_a, (n, 4), np.float32)[:, :2]
    ext = ctx.download(f.aabb, (n, 2), np.float32)
    rad = ctx.download(f.radii, (n,), np.int32)
    dep = ctx.download(f.depths, (n,), np.float32)
    t, F = np.array([tiles_x, tiles_y]), np.float32
    vis = rad > 0
    c, r = xy[vis] / F(16), ext[vis] / F(16)
    lo = np.clip((c - r).astype(np.int64), 0, t)  # truncated, as a float to int conversion
    hi = np.clip((c + r + F(1)).astype(np.int64), 0, t)
    ids = np.nonzero(vis)[0]
    order = np.lexsort((ids, dep[vis].view(np.uint32)))
    lists = [[] for _ in range(tiles_x * tiles_y)]
    for k in order:
        for y in range(lo[k, 1], hi[k, 1]):
            for x in range(lo[k, 0], hi[k, 0]):
                lists[y * tiles_x + x].append(ids[k])
    start = np.concatenate([[0], np.cumsum([len(v) for v in lists])])
    return start, np.array([g for v in lists for g in v], np.int64)


@pytest.mark.parametrize("W,H,n,scale", [
    (128, 128, 1, -2.0),      # one supertile, one record
    (128, 128, 63, -2.0), (128, 128, 64, -2.0), (128, 128, 65, -1.0),
    (16, 16, 300, -2.5),      # one tile
    (129, 128, 300, -2.0),    # nine tiles: the first view that takes both levels
    (145, 271, 700, -3.0),    # odd sizes, splats around a tile
    (1024, 1024, 500, -2.5),  # exactly one level-1 node
    (1025, 1040, 500, -1.5),  # four nodes, three of them one tile wide
    (2070, 40, 400, -2.0),    # three nodes side by side
    (1030, 2060, 400, -2.0),  # six nodes: the first launches of their own for prefix and plan
    (640, 360, 5000, -4.0),   # several units per node
    (200, 150, 70000, -5.0),  # more entries than one group per wave holds at level 2
])
def test_lists_hold_each_tiles_gaussians_in_depth_order(W, H, n, scale):
    from msplat._abi import Context
    from msplat.backend import DeviceGaussians, render
    from msplat.camera import look_at, make_camera
    from msplat.scenes import random_scene
    ctx = Context(0)
    sc = random_scene(n + W, n, degree=0, log_scale=(scale, 0.6))
    if n > 64:  # equal depths: the id breaks the tie
        sc["means"][n // 2:] = sc["means"][:n - n // 2]
    cam = make_camera(look_at((2.2, 0.5, 2.4), (0, 0, 0)), W, H, 0.9 * max(W, H), 0.9 * max(W, H))
    dg = DeviceGaussians(ctx, sc)
    render(ctx, dg, cam, BG)
    f = ctx.frame()
    start, gids = _expected(ctx, f, n, cam["tiles_x"], cam["tiles_y"])
    assert f.num_isects == start[-1] == len(gids)
    np.testing.assert_array_equal(ctx.download(f.tile_start, (f.num_tiles + 1,), np.int32), start)
    np.testing.assert_array_equal(ctx.download(f.isect_gid, (len(gids),), np.int32), gids)
    ctx.close()


def test_lists_and_keys_at_street_scale():
    """475,115 gaussians at 1264x832 (4,108 tiles, two level-1 nodes, millions of
    intersections): the lists, their ranges, and the 64-bit (tile << 32 | depth bits) keys made
    of them, against the same restatement with the rectangles expanded whole."""
    from msplat._abi import FRAME_KEYS64, Context
    from msplat.backend import DeviceGaussians, render
    from msplat.scenes import street_cameras, street_points
    n, W, H = 475_115, 1264, 832
    ctx = Context(0)
    ctx.set_flags(FRAME_KEYS64)
    dg = DeviceGaussians.from_points(ctx, *street_points(0, n), degree=0)
    cam = street_cameras(4, W, H, 900.0, 900.0)[1]
    render(ctx, dg, cam, BG)
    f = ctx.frame()
    M, tx, ty = int(f.num_isects), cam["tiles_x"], cam["tiles_y"]
    F, t = np.float32, np.array([tx, ty])
    ids = np.nonzero(ctx.download(f.radii, (n,), np.int32) > 0)[0]
    dep = ctx.download(f.depths, (n,), np.float32).view(np.uint32)
    c = ctx.download(f.splat_a, (n, 4), np.float32)[ids, :2] / F(16)
    r = ctx.download(f.aabb, (n, 2), np.float32)[ids] / F(16)
    lo, hi = np.clip((c - r).astype(np.int64), 0, t), np.clip((c + r + F(1)).astype(np.int64), 0, t)
    order = np.lexsort((ids, dep[ids]))
    ids, lo, size = ids[order], lo[order], np.maximum(hi - lo, 0)[order]
    count = size[:, 0] * size[:, 1]
    at = np.repeat(np.arange(ids.size), count)
    k = np.arange(at.size) - np.repeat(np.cumsum(count) - count, count)
    tile = (lo[at, 1] + k // size[at, 0]) * tx + lo[at, 0] + k % size[at, 0]
    by_tile = np.argsort(tile, kind="stable")
    gids, tile = ids[at[by_tile]], tile[by_tile]
    assert M == gids.size > 1_000_000
    np.testing.assert_array_equal(ctx.download(f.tile_start, (tx * ty + 1,), np.int32),
                                  np.searchsorted(tile, np.arange(tx * ty + 1)))
    np.testing.assert_array_equal(ctx.download(f.isect_gid, (M,), np.int32), gids)
    np.testing.assert_array_equal(ctx.download(f.isect_keys, (M,), np.uint64),
                                  (tile.astype(np.uint64) << np.uint64(32)) | dep[gids].astype(np.uint64))
    ctx.close()


@pytest.mark.parametrize("graph", [False, True])
def test_batched_lists_give_the_one_view_images(graph):
    """Views of one to nine level-1 nodes in one batch (and one behind the camera): their
    images equal the one-view renders bit for bit, also after a smaller batch shrank the
    frame within buffers sized for more."""
    from msplat._abi import TUNE_CHUNKS, Context, DeviceArray
    from msplat.backend import (BatchViews, DeviceGaussians, adam_coeffs, render_batch_numpy, render_numpy,
                                train_step_batch)
    from msplat.camera import look_at, make_camera
    from msplat.scenes import random_scene
    ctx, one = Context(0), Context(0)
    one.set_tuning(TUNE_CHUNKS, 1)
    sc = random_scene(5, 3000, degree=1, log_scale=(-2.6, 0.7))
    dg = DeviceGaussians(ctx, sc)
    views = [(40, 30, (2.5, 0.6, 2.0)), (128, 128, (2.0, 0.0, 2.0)), (1025, 520, (2.4, 1.0, 1.5)),
             (2064, 2050, (1.9, 0.3, 2.2)), (333, 217, (-2.5, 0.2, 2.0))]
    cams = [make_camera(look_at(e, (0, 0, 0)), w, h, 0.8 * w, 0.8 * w, dtu=1) for w, h, e in views]
    cams.append(make_camera(look_at((2.5, 0.0, 2.5), (5.0, 0.0, 5.0)), 96, 64, 90.0, 90.0, dtu=1))
    for sub in (cams, cams[3:5], cams[:2], cams):
        if graph:  # the same sizes through a captured step first
            ctx.set_batch_graph(True)
            tg = [DeviceArray(ctx, (c["H"], c["W"], 3)) for c in sub]
            bv = BatchViews(sub, 1, [BG], tg)
            for t in (1, 2):
                train_step_batch(ctx, dg, bv, *adam_coeffs([0.0] * 6, t))
        got = render_batch_numpy(ctx, dg, BatchViews(sub, 1, [BG]))
        for c, img in zip(sub, got):
            np.testing.assert_array_equal(img, render_numpy(one, dg, c, BG))
    ctx.close()
    one.close()


def _one_tile_cloud(n):
    """Depths over three octaves and many ties; some gaussians behind the camera."""
    from msplat.scenes import random_scene
    rng = np.random.default_rng(n)
    sc = random_scene(n, n, degree=0, log_scale=(-3.0, 0.1))
    sc["means"] = (rng.normal(0, 0.02, (n, 3))).astype(np.float32)
    z = rng.uniform(-0.5, 9, n).astype(np.float32)
    z[n // 2:] = np.round(z[n // 2:], 2)  # equal depths: the id breaks the tie
    sc["means"][:, 2] += z
    return sc


@pytest.mark.parametrize("n", [1, 1023, 1024, 1025, 300_000, 2 << 20])
def test_depth_order_at_block_edges(n):
    """One tile holds every visible gaussian, in (depth bits, id) order: around one block of
    the sort, whose last pass writes the list entries, and with its larger blocks."""
    from msplat._abi import Context
    from msplat.backend import DeviceGaussians, render
    from msplat.camera import look_at, make_camera
    ctx = Context(0)
    cam = make_camera(look_at((0, 0, -1), (0, 0, 1)), 16, 16, 14.0, 14.0)
    dg = DeviceGaussians(ctx, _one_tile_cloud(n))
    for _ in range(2):
        render(ctx, dg, cam, BG)
        f = ctx.frame()
        rad, dep = ctx.download(f.radii, (n,), np.int32), ctx.download(f.depths, (n,), np.float32)
        c = ctx.download(f.splat_a, (n, 4), np.float32)[:, :2] / np.float32(16)
        r = ctx.download(f.aabb, (n, 2), np.float32) / np.float32(16)
        ids = np.nonzero((rad > 0) & np.all((c - r < 1) & (c + r + np.float32(1) >= 1), axis=1))[0]
        gids = ctx.download(f.isect_gid, (int(f.num_isects),), np.int32)
        np.testing.assert_array_equal(gids, ids[np.lexsort((ids, dep[ids].view(np.uint32)))])
    assert n == 1 or len(gids) > 0.8 * n
    ctx.close()
