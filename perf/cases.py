"""The work a user of this framework has it do, as cases that can be timed and compared:
train steps (one view, prior-guided, batched), renders (one view as the render server
runs them, batched), the autograd function, and the initialisation from points.

Scenes follow the framework's own recipes (msplat/scenes.py and bench.py): the street
cloud (depth log-uniform around two capture centres), the served 64-cluster cloud, and the
small object scene, with scales from the clouds' 3-nearest-neighbour spacing. Every state
owns its context, as a trainer or a render slot does.
"""
import ctypes as C
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "msplat-street_amd"))

from msplat._abi import TUNE_CHUNKS, Context, DeviceArray, check, lib  # noqa: E402
from msplat.autograd import rasterize  # noqa: E402
from msplat.backend import (KEYS, BatchViews, DeviceGaussians, adam_coeffs, render, render_batch, sh_bases,  # noqa: E402
                            train_step, train_step_batch)
from msplat.camera import look_at, make_camera  # noqa: E402
from msplat.prior import DevicePrior, train_step_prior  # noqa: E402

BG = (0.6130, 0.0101, 0.3984)
# The schedule's rates times 1e-3, as at the end of a fine-tuning run: thousands of passes
# leave the scene as it is, so that every pass does the same work.
RATES = [1e-3 * v for v in (1.6e-4, 5e-3, 1e-3, 2.5e-3, 1.25e-4, 5e-2)]
SSIM_WEIGHT = 0.2
VIEW_SIZES = ((640, 360), (1264, 832), (1920, 1080), (2560, 1440))  # of batched training
SERVED_SIZES = ((640, 360), (1280, 720))  # a served batch holds about one 1080p view of pixels


def listed():
    return [
        # one step of a small run: 20k gaussians, 128x128 views (few tiles: depth-chunked), launches and latency
        dict(name="train_128", kind="train", scene="object", n=20000, degree=1, dtu=1, W=128, H=128, grow=0.0),
        # odd sizes of a mid-size capture, SH degree 2
        dict(name="train_odd", kind="train", scene="street", n=183297, degree=2, dtu=2, W=997, H=613, grow=-0.2),
        # the street scene early in its schedule: initial splats, SH degree 0 in use (the benchmark's timed steps)
        dict(name="train_street", kind="train", scene="street", n=475115, degree=3, dtu=0, W=1264, H=832, grow=0.0),
        # the same scene late in it: smaller splats, every SH band in use
        dict(name="train_street_late", kind="train", scene="street", n=475115, degree=3, dtu=3, W=1264, H=832, grow=-0.5),
        # the street preset: depth, sky and fill priors, learned sky, exposure, scale cap
        dict(name="train_prior", kind="prior", scene="street", n=475115, degree=3, dtu=1, W=1264, H=832, grow=0.0),
        # one batched step (captured graph) of 8 views of mixed resolution
        dict(name="train_batch", kind="train_batch", scene="street", n=1000000, degree=3, dtu=3, views=8, grow=0.0),
        # requests of the render server, from its smallest to its largest view and scene
        dict(name="render_360p", kind="render", scene="cloud", n=500000, degree=3, dtu=3, W=640, H=360, grow=0.0),
        dict(name="render_1080p", kind="render", scene="cloud", n=2000000, degree=3, dtu=3, W=1920, H=1080, grow=0.0),
        dict(name="render_2160p", kind="render", scene="cloud", n=3000000, degree=3, dtu=3, W=3840, H=2160, grow=0.0),
        # requests of one scene that queued and are rendered together
        dict(name="render_batch", kind="render_batch", scene="cloud", n=1000000, degree=3, dtu=3, views=4, grow=0.0),
        # a differentiable render and its gradients inside somebody's torch program
        dict(name="autograd", kind="autograd", scene="object", n=100003, degree=3, dtu=3, W=801, H=599, grow=0.3),
        # a scene's initialisation from a point cloud (exact 3-NN scales)
        dict(name="init", kind="init", scene="street", n=475115, degree=3),
    ]


def draw(rng):
    def log_uniform(a, b):
        return int(round(math.exp(rng.uniform(math.log(a), math.log(b)))))

    kind = rng.choice(["train", "train", "train", "prior", "train_batch", "render", "render", "render", "render_batch",
                       "autograd", "init"])
    degree = rng.choice([0, 1, 2, 3, 3])
    c = dict(kind=kind, degree=degree, dtu=rng.randint(0, degree), grow=round(rng.uniform(-0.6, 0.1), 3))
    if kind in ("render", "render_batch"):
        c.update(scene="cloud", n=log_uniform(30000, 2500000), grow=0.0)
    else:
        c.update(scene=rng.choice(["street", "street", "object"]), n=log_uniform(10000, 500000))
    if kind == "train_batch":
        c.update(scene="street", views=rng.randint(2, 6))
    elif kind == "render_batch":
        c.update(views=rng.randint(2, 6))
    elif kind == "init":
        c.update(scene="street")
        del c["grow"], c["dtu"]
    else:
        px = math.exp(rng.uniform(math.log(128 * 128), math.log(2.1e6 if kind == "render" else 1.1e6)))
        aspect = rng.uniform(0.9, 1.9)
        c.update(W=max(33, int(math.sqrt(px * aspect))), H=max(33, int(math.sqrt(px / aspect))))
        if rng.random() < 0.5:
            c.update(W=c["W"] | 1, H=c["H"] | 1)
    return c


# ── inputs ───────────────────────────────────────────────────────────────────


def _scene(case, g):
    """Parameter groups in the reference layouts, made on the GPU from generator g."""
    n, degree, dev = case["n"], case["degree"], "cuda"

    def normal(*shape):
        return torch.randn(shape, generator=g, device=dev)

    grow = case.get("grow", 0.0)
    if case["scene"] == "street":  # two capture centres, depth log-uniform in [2, 60] m
        d = torch.nn.functional.normalize(normal(n, 3), dim=1)
        r = torch.exp(math.log(2.0) + math.log(30.0) * torch.rand(n, generator=g, device=dev))
        means = d * r[:, None]
        means[1::2, 0] += 10.0
        density = 0.5 * n / (4.0 * math.pi * math.log(30.0) * r ** 3)
        scales = (0.718 * density ** (-1.0 / 3.0)).log()[:, None] + 0.2 * normal(n, 3)
        opac = -2.2 + 0.8 * normal(n, 1)
    elif case["scene"] == "cloud":  # 64 clusters (sigma 0.5 m) in an 8 m box, opaque
        centre = 8.0 * torch.rand((64, 3), generator=g, device=dev) - 4.0
        off = 0.5 * normal(n, 3)
        means = centre[torch.randint(0, 64, (n,), generator=g, device=dev)] + off
        density = n / 64.0 / ((2.0 * math.pi) ** 1.5 * 0.125) * torch.exp(-2.0 * (off * off).sum(1))
        scales = (0.718 * density ** (-1.0 / 3.0)).log().clamp(max=-1.0)[:, None].expand(n, 3) + 0.1 * normal(n, 3)
        opac = 1.5 + normal(n, 1)
    else:  # the small object scene
        means = 2.0 * torch.rand((n, 3), generator=g, device=dev) - 1.0
        scales = -4.5 + 0.5 * normal(n, 3)
        opac = normal(n, 1)
    rest = 0.05 * normal(n, sh_bases(degree) - 1, 3)  # (n, 0, 3) at degree 0: nothing is stored
    return dict(means=means, scales=scales + grow, quats=torch.nn.functional.normalize(normal(n, 4), dim=1),
                dc=0.5 * normal(n, 3), rest=rest, opac=opac)


def _device_gaussians(ctx, case, g):
    sc = {k: v.cpu().numpy() for k, v in _scene(case, g).items()}
    return DeviceGaussians(ctx, dict(sc, degree=case["degree"]))


def _camera(case, rng, W, H):
    dtu = case["dtu"]
    if case["scene"] == "street":  # on the path through the two centres, any heading
        p, yaw = np.array([rng.uniform(-5.0, 15.0), 0.0, 0.0]), rng.uniform(0, 2 * np.pi)
        pose, f = look_at(p, p + np.array([np.cos(yaw), -0.1, np.sin(yaw)])), 900.0 * W / 1264.0
    elif case["scene"] == "cloud":  # on a sphere of radius 3-10 m around the scene
        d = rng.normal(size=3) * np.array([1.0, 0.4, 1.0])
        pose, f = look_at(d / np.linalg.norm(d) * rng.uniform(3.0, 10.0), (0, 0, 0)), 0.9 * W
    else:
        th = rng.uniform(0, 2 * np.pi)
        pose, f = look_at((4.0 * np.cos(th), 0.3, 4.0 * np.sin(th)), (0, 0, 0)), 120.0 / 128.0 * W
    return make_camera(pose, W, H, f, f, dtu=dtu)


def _target(g, W, H):
    """A photograph's stand-in: smooth colours with grain."""
    low = torch.rand((1, 3, H // 24 + 2, W // 24 + 2), generator=g, device="cuda")
    img = torch.nn.functional.interpolate(low, (H, W), mode="bilinear", align_corners=True)[0]
    return (img + 0.04 * torch.randn((3, H, W), generator=g, device="cuda")).clamp(0, 1).permute(1, 2, 0).contiguous()


def _view_sizes(case, rng):
    sizes = VIEW_SIZES if case["kind"] == "train_batch" else SERVED_SIZES
    return [sizes[k % len(sizes)] for k in rng.permutation(case["views"])]


def _prior(case, rng, cam):
    """The street preset's prior at half resolution: ground-plane depth with invalid
    samples, sky above the horizon, the vehicle's hood not kept, a 512x128 learned sky."""
    pw, ph = max(case["W"] // 2, 2), max(case["H"] // 2, 2)
    horizon = 0.5 * (float(cam["cy"]) - 0.1 * float(cam["fy"]))
    yy = np.mgrid[0:ph, 0:pw][0].astype(np.float32)
    below = yy - np.float32(horizon)
    depth = np.where(below > 0.5, np.minimum(0.8 * float(cam["fy"]) / np.maximum(below, 0.5), 80.0), 0.0)
    depth[rng.random((ph, pw)) < 0.02] = 0.0
    aux = np.zeros((ph, pw, 4), np.uint8)
    aux[..., 0] = rng.integers(120, 256, (ph, pw))
    aux[..., 1] = np.where(below < -4.0, 255, 0)
    aux[..., 2] = np.where(yy < 0.94 * ph, 255, 0)
    sky = rng.uniform(0.3, 0.9, (128, 512, 3)).astype(np.float32)
    ident = np.zeros((8, 12), np.float32)
    ident[:, [0, 4, 8]] = 1.0
    bc2 = float(np.sqrt(np.float32(1 - 0.999)))
    return dict(aux=True, sky=True, sky_tex=sky, sky_grad=np.zeros_like(sky), sky_m1=np.zeros_like(sky),
                sky_m2=np.zeros_like(sky), sky_frame=(0, 1, 0, 1, 0, 0, 0, 0, -1), sky_step=1e-4, sky_bc2=bc2,
                prior_depth=depth.astype(np.float32), prior_aux=aux, has_depth=True, has_sky_mask=True, depth_weight=0.2,
                sky_weight=0.05, fill_weight=0.01, huber_delta=0.05, min_alpha=0.25, mask_photometric=True,
                exposure=True, cam_index=3, expo_params=ident, expo_m1=np.zeros_like(ident),
                expo_m2=np.zeros_like(ident), expo_grad=np.zeros(12, np.float32), expo_step=5e-5, expo_bc2=bc2,
                expo_reg=1e-2, log_max_scale_ratio=float(np.log(np.float32(10.0))), loss_terms=np.zeros(4, np.float32))


def _points_rgb(case, g):
    means = _scene(case, g)["means"]
    return means, torch.randint(0, 256, (case["n"], 3), generator=g, device="cuda", dtype=torch.uint8)


class State:
    """What a user's program keeps between calls."""


_stream = []


def _training_stream():
    if not _stream:
        _stream.append(torch.cuda.Stream())
    return _stream[0].cuda_stream


def prepare(case, seed):
    g = torch.Generator(device="cuda").manual_seed(1000 + int(seed))
    rng = np.random.default_rng(1000 + int(seed))
    s, kind = State(), case["kind"]
    s.case = case
    if kind == "autograd":
        s.params = {k: v.contiguous().requires_grad_(True) for k, v in _scene(case, g).items()}
        s.cam = _camera(case, rng, case["W"], case["H"])
        s.v_img = torch.randn((case["H"], case["W"], 3), generator=g, device="cuda")
        torch.cuda.synchronize()
        return s
    s.ctx = Context(0) if kind in ("render", "render_batch") else Context(0, _training_stream())
    if kind == "init":
        means, rgb = _points_rgb(case, g)
        s.dg = DeviceGaussians(s.ctx, dict(means=means.cpu().numpy(), degree=0, **{
            k: np.zeros((case["n"], w), np.float32) for k, w in (("scales", 3), ("quats", 4), ("dc", 3), ("rest", 3),
                                                                 ("opac", 1))}))
        s.rgb = DeviceArray.from_numpy(s.ctx, rgb.cpu().numpy())
        s.seed = int(seed)
        s.ctx.sync()
        return s
    s.dg = _device_gaussians(s.ctx, case, g)
    if kind in ("render", "render_batch"):
        s.ctx.set_tuning(TUNE_CHUNKS, 1)  # as the render server's slots do
    if kind in ("train_batch", "render_batch"):
        s.cams = [_camera(case, rng, w, h) for w, h in _view_sizes(case, rng)]
        s.pixels = sum(c["W"] * c["H"] for c in s.cams)
        targets = None
        if kind == "train_batch":  # the batch-size rule: rates x sqrt(V), decays to the power V
            targets = [DeviceArray.from_numpy(s.ctx, _target(g, c["W"], c["H"]).cpu().numpy()) for c in s.cams]
            V = len(s.cams)
            s.betas = (0.9 ** V, 0.999 ** V)
            s.adam = adam_coeffs([math.sqrt(V) * v for v in RATES], 1, *s.betas)
            s.ctx.set_batch_graph(True)
        s.views = BatchViews(s.cams, case["degree"], [BG], targets)
    else:
        s.cam = _camera(case, rng, case["W"], case["H"])
        s.pixels = case["W"] * case["H"]
        if kind in ("train", "prior"):
            s.gt = DeviceArray.from_numpy(s.ctx, _target(g, case["W"], case["H"]).cpu().numpy())
            s.adam = adam_coeffs(RATES, 1)
        if kind == "prior":
            s.prior = DevicePrior(s.ctx, _prior(case, rng, s.cam))
    if kind in ("render", "render_batch"):
        s.rgba = DeviceArray(s.ctx, (s.pixels, 4), np.uint8)
    s.ctx.sync()
    torch.cuda.synchronize()
    return s


# ── the passes ───────────────────────────────────────────────────────────────


class _Memory:
    """Device memory the framework owns, as the tensor library reads it; keeps the state."""

    def __init__(self, state, ptr, shape, dtype):
        self.state = state
        self.__cuda_array_interface__ = dict(shape=tuple(int(v) for v in shape), typestr=np.dtype(dtype).str,
                                             data=(int(ptr), False), version=2)


def _tensor(state, ptr, shape, dtype=np.float32):
    return torch.as_tensor(_Memory(state, ptr, shape, dtype), device="cuda")


def _trained(s):
    """The state of the scene after a step: parameters, moments, statistics."""
    if not hasattr(s, "views_of"):
        dg, n = s.dg, s.dg.n
        out = {}
        for name, group in (("p", dg.params), ("m1", dg.m1), ("m2", dg.m2)):
            for k in KEYS:
                if k != "rest" or dg.rest_bases:
                    out[name + "_" + k] = _tensor(None, group[k].ptr, (n, dg.widths[k]))
        for k in ("vis", "gn", "ms"):
            out[k] = _tensor(None, getattr(dg, k).ptr, (n,))
        s.views_of = out
    out = dict(s.views_of)
    out["p_opac"] = _tensor(s, s.dg.params["opac"].ptr, (s.dg.n, 1))  # keeps the state with the outputs
    return out


def run(s):
    kind = s.case["kind"]
    if kind == "train":
        train_step(s.ctx, s.dg, s.cam, BG, s.gt, *s.adam, ssim_weight=SSIM_WEIGHT, read_loss=False)
        return _trained(s)
    if kind == "prior":
        train_step_prior(s.ctx, s.dg, s.cam, BG, s.gt, *s.adam, s.prior, ssim_weight=SSIM_WEIGHT, read_loss=False)
        out = _trained(s)
        for k in ("sky_tex", "sky_m1", "sky_m2", "expo_params", "expo_m1", "expo_m2", "loss_terms"):
            out[k] = _tensor(None, s.prior.arrays[k].ptr, s.prior.shapes[k])
        return out
    if kind == "train_batch":
        losses = train_step_batch(s.ctx, s.dg, s.views, *s.adam, SSIM_WEIGHT, *s.betas)
        return dict(_trained(s), losses=losses)
    if kind == "render":
        img = render(s.ctx, s.dg, s.cam, BG)
        check(lib().msplat_hip_pack_rgba8(s.ctx.ptr, C.c_void_p(img), s.pixels, C.c_void_p(s.rgba.ptr)))
        return dict(image=_tensor(s, img, (s.pixels, 3)), rgba=_tensor(s, s.rgba.ptr, (s.pixels, 4), np.uint8))
    if kind == "render_batch":
        img, _ = render_batch(s.ctx, s.dg, s.views)
        check(lib().msplat_hip_pack_rgba8(s.ctx.ptr, C.c_void_p(img), s.pixels, C.c_void_p(s.rgba.ptr)))
        return dict(image=_tensor(s, img, (s.pixels, 3)), rgba=_tensor(s, s.rgba.ptr, (s.pixels, 4), np.uint8))
    if kind == "autograd":
        img = rasterize(*(s.params[k] for k in KEYS), s.cam, BG)
        grads = torch.autograd.grad(img, [s.params[k] for k in KEYS if k != "rest" or s.case["degree"]], s.v_img)
        names = [k for k in KEYS if k != "rest" or s.case["degree"]]
        return dict(image=img.detach(), **{"g_" + k: v for k, v in zip(names, grads)})
    p, n = s.dg.params, s.dg.n
    check(lib().msplat_hip_init_gaussians(s.ctx.ptr, p["means"].ptr, s.rgb.ptr, n, s.seed, math.log(0.1 / 0.9),
                                          p["scales"].ptr, p["quats"].ptr, p["dc"].ptr, p["opac"].ptr))
    return {k: _tensor(s, p[k].ptr, (n, w)) for k, w in (("scales", 3), ("quats", 4), ("dc", 3), ("opac", 1))}


# ── what a pass cannot do without ────────────────────────────────────────────


def _pixels(case):
    if "views" not in case:
        return case["W"] * case["H"]
    sizes = VIEW_SIZES if case["kind"] == "train_batch" else SERVED_SIZES
    return sum(w * h for w, h in (sizes[k % len(sizes)] for k in range(case["views"])))


def work(case):
    n, kind = case["n"], case["kind"]
    if kind == "init":  # points and colours in, scales, quaternions, DC and opacity out
        return dict(bytes=n * (15 + 44), flops=200.0 * n)
    px = _pixels(case)
    # gaussians in view (about a sixth of a street scene), their SH floats in use
    seen = n if case["scene"] != "street" else n * min(1.0, 0.17 * (1 if "views" not in case else 0.5 * case["views"]))
    sh = 3 * sh_bases(case["dtu"])
    composited = 40.0 * px  # pixel-gaussian pairs that reach a pixel
    fwd = dict(bytes=4.0 * (11 * n + sh * seen) + 12.0 * px, flops=250.0 * n + 20.0 * composited)
    if kind in ("render", "render_batch"):
        return dict(bytes=fwd["bytes"] + 4.0 * px, flops=fwd["flops"])
    if kind == "autograd":  # the upstream gradient in, six gradients out
        return dict(bytes=fwd["bytes"] + 12.0 * px + 4.0 * n * (11 + 3 * sh_bases(case["degree"])),
                    flops=fwd["flops"] + 400.0 * n + 50.0 * composited)
    # the target in; parameters out, both moments in and out (dense groups over every
    # gaussian, SH over the seen ones), three statistics in and out
    return dict(bytes=4.0 * (11 * n + sh * seen) * 6 + 24.0 * seen + 12.0 * px,
                flops=fwd["flops"] + 500.0 * n + 50.0 * composited + 800.0 * px)


def tolerance(case):
    # About four times what the 32-bit results differ from 64-bit ones by over the declared
    # ranges. Most of it is single pixels where a pair sits on a cut-off (alpha 1/255,
    # sigma 5.55, transmittance 1e-4) and falls on its other side.
    kind = case["kind"]
    if kind == "init":
        return dict(rel=5e-7, max=2e-6)
    if kind in ("render", "render_batch"):
        return dict(rel=2e-5, max=0.01, differ=1e-3)
    return dict(rel=4e-3, max=0.5)


# ── the same results in 64 bits, in plain torch ──────────────────────────────

SH = dict(c0=0.28209479177387814, c1=0.4886025119029199)


def _sh_basis(d, degree):
    x, y, z = d.unbind(1)
    xx, yy, zz, xy, yz, xz = x * x, y * y, z * z, x * y, y * z, x * z
    b = [torch.full_like(x, SH["c0"])]
    if degree >= 1:
        b += [-SH["c1"] * y, SH["c1"] * z, -SH["c1"] * x]
    if degree >= 2:
        b += [1.0925484305920792 * xy, -1.0925484305920792 * yz, 0.31539156525252005 * (2 * zz - xx - yy),
              -1.0925484305920792 * xz, 0.5462742152960396 * (xx - yy)]
    if degree >= 3:
        b += [-0.5900435899266435 * y * (3 * xx - yy), 2.890611442640554 * xy * z,
              -0.4570457994644658 * y * (4 * zz - xx - yy), 0.3731763325901154 * z * (2 * zz - 3 * xx - 3 * yy),
              -0.4570457994644658 * x * (4 * zz - xx - yy), 1.445305721320277 * z * (xx - yy),
              -0.5900435899266435 * x * (xx - 3 * yy)]
    return torch.stack(b, 1)


def _project(p, cam, dtu):
    """Pixel centres, conics, raw colours, opacities, depths, tile rectangles, radii (64 bits)."""
    f64 = dict(dtype=torch.float64, device="cuda")
    vm = torch.tensor(np.asarray(cam["viewmat"], np.float64).reshape(4, 4), **f64)
    pm = torch.tensor(np.asarray(cam["projmat"], np.float64).reshape(4, 4), **f64)
    fx, fy, cx, cy, W, H = (float(cam[k]) for k in ("fx", "fy", "cx", "cy", "W", "H"))
    m = p["means"]
    pv = m @ vm[:3, :3].T + vm[:3, 3]
    z = pv[:, 2]
    front = z > 0.01
    zs = torch.where(front, z, torch.ones_like(z))
    lim = torch.tensor([1.3 * 0.5 * W / fx, 1.3 * 0.5 * H / fy], **f64)
    xy_c = pv[:, :2] + ((pv[:, :2] / zs[:, None]).clamp(-lim, lim) * zs[:, None] - pv[:, :2]).detach()
    q = torch.nn.functional.normalize(p["quats"], dim=1)
    w, x, y, zq = q.unbind(1)
    R = torch.stack([1 - 2 * (y * y + zq * zq), 2 * (x * y - w * zq), 2 * (x * zq + w * y),
                     2 * (x * y + w * zq), 1 - 2 * (x * x + zq * zq), 2 * (y * zq - w * x),
                     2 * (x * zq - w * y), 2 * (y * zq + w * x), 1 - 2 * (x * x + y * y)], 1).view(-1, 3, 3)
    M = R * torch.exp(p["scales"])[:, None, :]
    rz = 1.0 / zs
    t0 = fx * rz[:, None] * vm[0, :3] - (fx * xy_c[:, 0] * rz * rz)[:, None] * vm[2, :3]
    t1 = fy * rz[:, None] * vm[1, :3] - (fy * xy_c[:, 1] * rz * rz)[:, None] * vm[2, :3]
    u0, u1 = (M * t0[:, :, None]).sum(1), (M * t1[:, :, None]).sum(1)
    a, b, c = (u0 * u0).sum(1) + 0.3, (u0 * u1).sum(1), (u1 * u1).sum(1) + 0.3
    det = a * c - b * b
    conic = torch.stack([c / det, -b / det, a / det], 1)
    h = m @ pm[:, :3].T + pm[:, 3]
    rw = 1.0 / (torch.where(front, h[:, 3], torch.ones_like(z)) + 1e-6)
    xy = torch.stack([0.5 * W * h[:, 0] * rw + cx - 0.5, 0.5 * H * h[:, 1] * rw + cy - 0.5], 1)
    pos = torch.tensor(np.asarray(cam["cam_pos"], np.float64), **f64)
    basis = _sh_basis(torch.nn.functional.normalize((m - pos).detach(), dim=1), dtu)
    coef = torch.cat([p["dc"][:, None, :], p["rest"]], 1)[:, :basis.shape[1]]
    rgb = (coef * basis[:, :, None]).sum(1)
    opac = torch.sigmoid(p["opac"].reshape(-1))
    with torch.no_grad():
        tx, ty = int(cam["tiles_x"]), int(cam["tiles_y"])
        rx, ry = torch.ceil(3 * a.sqrt()), torch.ceil(3 * c.sqrt())
        lo = lambda v, r, t: ((v - r) / 16).trunc().clamp(0, t).long()  # noqa: E731
        hi = lambda v, r, t: ((v + r) / 16 + 1).trunc().clamp(0, t).long()  # noqa: E731
        big = 1e9
        vx, vy = xy[:, 0].clamp(-big, big), xy[:, 1].clamp(-big, big)
        x0, x1, y0, y1 = lo(vx, rx, tx), hi(vx, rx, tx), lo(vy, ry, ty), hi(vy, ry, ty)
        count = torch.where(front & (det != 0), (x1 - x0).clamp(min=0) * (y1 - y0).clamp(min=0), torch.zeros_like(x0))
        # the list order is that of the 32-bit depths, each product and sum rounded
        v32, m32 = np.asarray(cam["viewmat"], np.float32).reshape(4, 4)[2], m.float()
        z32 = m32[:, 0] * float(v32[0]) + m32[:, 1] * float(v32[1])
        z32 = z32 + m32[:, 2] * float(v32[2])
        z32 = z32 + float(v32[3])
    return xy, conic, rgb, opac, z32, (x0, y0, x1 - x0, count)


def _tile_lists(z, rect, tiles_x, ntiles):
    x0, y0, w, count = rect
    order = torch.argsort(z, stable=True)
    order = order[count[order] > 0]
    c = count[order]
    ids = torch.repeat_interleave(order, c)
    k = torch.arange(ids.numel(), device="cuda") - torch.repeat_interleave(c.cumsum(0) - c, c)
    tile = (y0[ids] + k // w[ids]) * tiles_x + x0[ids] + k % w[ids]
    tile, at = torch.sort(tile.int(), stable=True)
    start = torch.searchsorted(tile, torch.arange(ntiles + 1, device="cuda", dtype=torch.int32))
    return ids[at], start


def _tile_chunks(start, budget):
    """Groups of tiles of like list length with at most `budget` padded pairs each."""
    length = (start[1:] - start[:-1]).cpu().numpy()
    order = [int(t) for t in np.argsort(-length, kind="stable") if length[t] > 0]
    at = 0
    while at < len(order):
        L = int(length[order[at]])
        k = max(1, budget // (L * 256))
        yield torch.tensor(order[at:at + k], device="cuda"), L
        at += k


def _composite(tiles, L, ids, start, cam, xy, conic, rgb, opac):
    """Colour sums [t, 256, 3], final transmittance [t, 256] and pixel ids of some tiles."""
    W, H, tx = int(cam["W"]), int(cam["H"]), int(cam["tiles_x"])
    k = torch.arange(L, device="cuda")
    at = start[tiles][:, None] + k
    real = at < start[tiles + 1][:, None]
    gid = ids[at.clamp(max=ids.numel() - 1)]
    j = torch.arange(256, device="cuda")
    px, py = (tiles % tx)[:, None] * 16 + j % 16, (tiles // tx)[:, None] * 16 + j // 16
    inside = (px < W) & (py < H)
    d = xy[gid]
    dx, dy = d[:, :, None, 0] - px[:, None, :], d[:, :, None, 1] - py[:, None, :]
    cn = conic[gid]
    sigma = 0.5 * (cn[:, :, 0, None] * dx * dx + cn[:, :, 2, None] * dy * dy) + cn[:, :, 1, None] * dx * dy
    del dx, dy
    al = opac[gid][:, :, None] * torch.exp(-sigma)
    al = torch.clamp(al, max=0.999)
    ok = real[:, :, None] & (sigma >= 0) & (sigma < 5.55) & (al >= 1.0 / 255.0)
    al = torch.where(ok, al, torch.zeros_like(al))
    del sigma
    logs = torch.log1p(-al)
    incl = logs.cumsum(1)
    ok = ok & (incl.detach() > math.log(1e-4))  # until the transmittance would fall to 1e-4
    weight = torch.where(ok, al * torch.exp(incl - logs), torch.zeros_like(al))
    colour = (rgb[gid] + 0.5).clamp(min=0)
    out = torch.bmm(weight.transpose(1, 2).contiguous(), colour.contiguous())
    T = torch.exp(torch.where(ok, logs, torch.zeros_like(logs)).sum(1))
    return out, T, torch.where(inside, py * W + px, torch.full_like(px, -1))


def _exact_image(cam, proj, budget=24_000_000):
    xy, conic, rgb, opac, z, rect = proj
    W, H = int(cam["W"]), int(cam["H"])
    ids, start = _tile_lists(z, rect, int(cam["tiles_x"]), int(cam["tiles_x"]) * int(cam["tiles_y"]))
    bg = torch.tensor(np.asarray(BG, np.float32).astype(np.float64), device="cuda")
    img = bg.expand(W * H, 3).clone()
    with torch.no_grad():
        for tiles, L in _tile_chunks(start, budget):
            out, T, pid = _composite(tiles, L, ids, start, cam, xy, conic, rgb, opac)
            keep = pid >= 0
            img[pid[keep]] = (out + T[:, :, None] * bg)[keep]
    return img, ids, start


def _exact_gradients(cam, p, dtu, v_of_image):
    """(image, v_of_image's own result, |dL/dxy|) with the gradients accumulated into p's leaves."""
    proj = _project(p, cam, dtu)
    two = [t.detach().requires_grad_(True) for t in proj[:4]]
    img, ids, start = _exact_image(cam, [t.detach() for t in proj[:4]] + list(proj[4:]))
    extra, v = v_of_image(img.clamp(0, 1))
    bg = torch.tensor(np.asarray(BG, np.float32).astype(np.float64), device="cuda")
    for tiles, L in _tile_chunks(start, 12_000_000):
        out, T, pid = _composite(tiles, L, ids, start, cam, *two)
        vt = torch.where((pid >= 0)[:, :, None], v[pid.clamp(min=0)], torch.zeros((), dtype=v.dtype, device="cuda"))
        torch.autograd.backward([out, T], [vt, (vt * bg).sum(2)])
    seen = proj[5][3] > 0
    grads = [torch.zeros_like(t) if t.grad is None else t.grad for t in two]
    torch.autograd.backward(list(proj[:4]), [torch.where(seen.view(-1, *[1] * (g.dim() - 1)), g, torch.zeros_like(g))
                                             for g in grads])
    return img.clamp(0, 1), extra, torch.where(seen, grads[0].norm(dim=1), torch.zeros_like(grads[0][:, 0])), seen


def _exact_loss(gt, W, H):
    """0.8 L1 + 0.2 (1 - SSIM), 11-tap gaussian window over zero padding, and its gradient."""
    g1 = torch.tensor([0.0010283801, 0.0075987581, 0.0360007721, 0.1093606895, 0.2130055377, 0.2660117249, 0.2130055377,
                       0.1093606895, 0.0360007721, 0.0075987581, 0.0010283801], dtype=torch.float64, device="cuda")

    def blur(t):
        for dim, shape in ((2, (H, 1)), (3, (1, W))):
            pad = [0, 0, 5, 5] if dim == 2 else [5, 5, 0, 0]
            tp = torch.nn.functional.pad(t, pad)
            t = sum(g1[k] * tp.narrow(dim, k, t.shape[dim]) for k in range(11))
        return t

    y = gt.double().permute(2, 0, 1)[None]

    def of(img):
        x = img.view(H, W, 3).permute(2, 0, 1)[None].detach().requires_grad_(True)
        mx, my = blur(y), blur(x)
        vx, vy, cxy = blur(y * y) - mx * mx, blur(x * x) - my * my, blur(x * y) - mx * my
        ssim = ((2 * mx * my + 1e-4) * (2 * cxy + 9e-4)) / ((mx * mx + my * my + 1e-4) * (vx + vy + 9e-4))
        loss = SSIM_WEIGHT * (1 - ssim.mean()) + (1 - SSIM_WEIGHT) * (y - x).abs().mean()
        loss.backward()
        return loss.item(), x.grad[0].permute(1, 2, 0).reshape(-1, 3)

    return of


def _leaves(case, g):
    return {k: v.double().contiguous().requires_grad_(True) for k, v in _scene(case, g).items()}


def exact(case, seed):
    kind = case["kind"]
    if kind == "prior":
        return None
    g = torch.Generator(device="cuda").manual_seed(1000 + int(seed))
    rng = np.random.default_rng(1000 + int(seed))
    if kind == "init":
        means, rgb = _points_rgb(case, g)
        n, m = case["n"], means.double()
        out = torch.empty(n, dtype=torch.float64, device="cuda")
        for i in range(0, n, 512):  # coordinate differences: no cancellation of squared norms
            d2 = sum((m[i:i + 512, None, a] - m[None, :, a]) ** 2 for a in range(3))
            out[i:i + 512] = d2.topk(4, dim=1, largest=False).values[:, 1:].sqrt().mean(1)
        return dict(scales=out.log()[:, None].expand(n, 3), quats=None,
                    dc=(rgb.double() / 255.0 - 0.5) / SH["c0"],
                    opac=torch.full((n, 1), math.log(0.1 / 0.9), dtype=torch.float64))
    if case["n"] * (case["views"] if kind == "train_batch" else 1) > 2500000:  # too long in 64 bits
        return None
    p = _leaves(case, g)
    if kind in ("render", "render_batch"):
        cams = [_camera(case, rng, w, h) for w, h in _view_sizes(case, rng)] if kind == "render_batch" else \
            [_camera(case, rng, case["W"], case["H"])]
        with torch.no_grad():
            img = torch.cat([_exact_image(c, _project(p, c, case["dtu"]))[0] for c in cams]).clamp(0, 1)
        return dict(image=img, rgba=None)
    if kind == "autograd":
        cam = _camera(case, rng, case["W"], case["H"])
        v = torch.randn((case["H"], case["W"], 3), generator=g, device="cuda").double().view(-1, 3)
        img = _exact_gradients(cam, p, case["dtu"], lambda _: (None, v))[0]
        return dict(image=img.view(case["H"], case["W"], 3), **{"g_" + k: p[k].grad if p[k].grad is not None else
                    torch.zeros_like(p[k]) for k in KEYS if k != "rest" or case["degree"]})
    if kind == "train_batch":
        cams = [_camera(case, rng, w, h) for w, h in _view_sizes(case, rng)]
        beta1, beta2 = 0.9 ** len(cams), 0.999 ** len(cams)
        rates = [math.sqrt(len(cams)) * v for v in RATES]
    else:
        cams, beta1, beta2, rates = [_camera(case, rng, case["W"], case["H"])], 0.9, 0.999, RATES
    start = {k: v.detach().clone() for k, v in p.items()}
    gn, losses, any_seen = 0.0, [], False
    for c in [(c, _target(g, c["W"], c["H"])) for c in cams]:
        _, loss, norm, seen = _exact_gradients(c[0], p, case["dtu"], _exact_loss(c[1], c[0]["W"], c[0]["H"]))
        gn, any_seen = gn + norm, any_seen | seen
        losses.append(loss)
    out = {}
    for i, k in enumerate(KEYS):
        if k == "rest" and not case["degree"]:
            continue
        grad = p[k].grad if p[k].grad is not None else torch.zeros_like(p[k])
        m1, m2 = (1 - beta1) * grad, (1 - beta2) * grad * grad
        out["m1_" + k], out["m2_" + k] = (t.reshape(case["n"], -1) for t in (m1, m2))
        step = rates[i] / (1 - beta1) * m1 / (m2.sqrt() / math.sqrt(1 - beta2) + 1e-8)
        out["p_" + k] = (start[k] - step).reshape(case["n"], -1)
    out.update(vis=None, gn=gn, ms=None)
    if kind == "train_batch":
        out["losses"] = torch.tensor(losses, dtype=torch.float64)
    return out
