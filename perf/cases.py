"""The workloads whose speed is tracked, each through a public entry point.

A case is a dict of plain values; "kind" names the call:

  frame      one frame of the SSVGI renderer (lgx_renderer_render, eager: a
             moving camera declares its passes anew every frame): pyramids,
             pre-blur, horizon gather, interleave, denoise, composite
  target     the many-direction gather of one crop of a frame, as the training
             pairs of the denoiser are made (lgx_gather with a region)
  pyramid    Hi-Z and radiance mips with the pre-blur (lgx_mip_build,
             lgx_box_blur)
  bilateral  one pass of the geometry-aware filter (lgx_bilateral)
  denoise    the U-Net from a G-buffer and a noisy image (lgx_unet_denoise)
  forward    the U-Net on a batch of input records (lgx_unet_forward)
  backward   forward, loss and gradients of one training batch, the gradients
             read back as a data-parallel trainer does (lgx_unet_backward,
             lgx_unet_get_state)
  batch      the noisy gathers of several views of uneven size
             (lgx_batch_run without a network)

prepare() makes inputs from the seed alone: a room with boxes and spheres,
ray cast here into a G-buffer, and the handles a program keeps (renderer,
network with its autotuned tiles, batch).  exact() restates each path in
64-bit torch.
"""
import ctypes as C
import json
import math

import numpy as np
import torch

from legitengine_amd import denoiser as dn
from legitengine_amd import device as dev
from legitengine_amd import lgx

PI = float(np.float32(3.1415))  # the shader's constant
AMBIENT = float(np.float32(0.01))
LAYERS = [(9, 32), (32, 32), (32, 64), (64, 64), (64, 128), (128, 128), (192, 64), (64, 64), (96, 32), (32, 32)]


# ------------------------------------------------------------------ the cases

def _frame(name, w, h, fmt, dirs, steps, levels, **kw):
    c = dict(kind="frame", w=w, h=h, fmt=fmt, dirs=dirs, steps=steps, levels=levels, sampler="hiz", grid=4,
             footprint=0, passes=2, radius=4, composite=False, tile=0)
    c.update(kw)
    return dict(c, name=name) if name else c


def listed():
    return [
        # the smallest frame: a thumbnail or probe view, where launches and latency count
        _frame("frame_256", 256, 256, "f32", 16, 32, 5),
        # the ordinary frame of an application, with the launch shape its start-up tuning picks
        _frame("frame_1080p", 1920, 1080, "mixed", 32, 64, 6, tile=4),
        # a window resized by hand: extents the pattern does not divide, few directions, lit image out
        _frame("frame_1279x719", 1279, 719, "f32", 8, 64, 6, radius=3, composite=True),
        # the shader's own mode: trilinear samples of averaged, pre-blurred pyramids, no step cap
        _frame("reference_1080p", 1920, 1080, "mixed", 4, 0, 10, sampler="trilinear", passes=1, composite=True),
        # the learned denoiser's input: four directions of a 256-direction march on an 8x8 pattern
        _frame("noisy_1080p", 1920, 1080, "mixed", 4, 0, 6, grid=8, footprint=256, passes=0, tile=28),
        # the denoiser's training target of one crop: 256 directions, summed in double
        dict(name="target_crop", kind="target", w=1920, h=1080, crop=256, dirs=256, precision="acc64", levels=6),
        # pyramids of a 4K G-buffer
        dict(name="pyramid_2160p", kind="pyramid", w=3840, h=2160, fmt="mixed", levels=6, sampler="hiz"),
        # one denoise pass of a 1440p frame
        dict(name="bilateral_1440p", kind="bilateral", w=2560, h=1440, fmt="mixed", radius=4),
        # the learned denoiser on a frame
        dict(name="denoise_1080p", kind="denoise", w=1920, h=1080, fmt="mixed"),
        # scoring a batch of crops (validation, hard-example selection)
        dict(name="forward_16x256", kind="forward", n=16, w=256, h=256),
        # the training batch
        dict(name="backward_16x256", kind="backward", n=16, w=256, h=256, loss="l2"),
        # several clients' views in one submission, one of each size that is served
        dict(name="batch_4", kind="batch", views="512x512,1280x720,1920x1080,2560x1440", tile=28),
    ]


def _cost(c):
    w = work(c)
    return max(w["bytes"], w["flops"] / 50)


def _draw(rng):
    def log(a, b):
        return int(round(math.exp(rng.uniform(math.log(a), math.log(b)))))

    def extent(lo=160, hi=2560):
        w = log(lo, hi)
        return w, max(96, int(w * rng.choice([0.5625, 0.625, 0.75, 1.0])) + rng.randrange(3))

    kind = rng.choice(["frame", "frame", "frame", "target", "pyramid", "bilateral", "denoise", "forward", "backward",
                       "batch"])
    fmt = rng.choice(["f32", "mixed", "mixed"])
    if kind == "frame":
        w, h = extent()
        mode = rng.choice(["plain", "plain", "reference", "noisy"])
        if mode == "plain":
            return _frame(None, w, h, fmt, rng.choice([8, 12, 16, 24, 32]), rng.choice([32, 64]), rng.choice([4, 5, 6]),
                          radius=rng.choice([2, 3, 4]), composite=rng.random() < 0.5, tile=rng.choice([0, 4]))
        if mode == "reference":
            return _frame(None, w, h, fmt, 4, 0, rng.choice([5, 6]), sampler="trilinear", passes=1, composite=True)
        return _frame(None, w, h, fmt, 4, 0, rng.choice([5, 6]), grid=8, footprint=256, passes=0, tile=28)
    if kind == "target":
        return dict(kind="target", w=1920, h=1080, crop=rng.choice([64, 96, 128, 200, 256]), dirs=rng.choice([64, 128, 192, 256]),
                    precision=rng.choice(["acc64", "acc64", "f64"]), levels=6)
    if kind == "pyramid":
        w, h = extent(160, 3840)
        return dict(kind="pyramid", w=w, h=h, fmt=fmt, levels=rng.choice([4, 5, 6]),
                    sampler=rng.choice(["hiz", "hiz", "trilinear"]))
    if kind == "bilateral":
        w, h = extent()
        return dict(kind="bilateral", w=w, h=h, fmt=fmt, radius=rng.choice([2, 3, 4, 6]))
    if kind == "denoise":
        w, h = extent()
        return dict(kind="denoise", w=w // 4 * 4, h=h // 4 * 4, fmt=fmt)
    if kind in ("forward", "backward"):
        c = dict(kind=kind, n=rng.randrange(1, 17), w=4 * log(16, 64), h=4 * log(16, 64))
        return dict(c, loss=rng.choice(["l1", "l2"])) if kind == "backward" else c
    views = []
    for _ in range(rng.randrange(2, 5)):
        views.append("%dx%d" % extent(256, 1600))
    return dict(kind="batch", views=",".join(views), tile=28)


def draw(rng):
    top = max(_cost(c) for c in listed())
    while True:
        c = _draw(rng)
        if _cost(c) <= top:
            return c


# ------------------------------------------------------------- what they need

def _steps(w, footprint, cap):
    """Mean on-screen steps of a march: the offsets grow by 2 pi / F + 1 from w / 1000 to about 0.35 w."""
    s = math.log(350.0) / math.log(2 * PI / footprint + 1)
    return min(s, cap) if cap > 0 else s


def _gather_flops(px, w, dirs, footprint, cap):
    # a step: position 4, texel 6, delta 10, horizon test 5, a tenth of a hit's 60; a direction's set-up 200
    return px * dirs * (_steps(w, footprint or dirs, cap) * 31.0 + 200.0)


def _unet_flops(px):
    s = [1, 1, 4, 4, 16, 16, 4, 4, 1, 1]
    return px * (sum(18.0 * ci * co / k for (ci, co), k in zip(LAYERS, s)) + 2 * 96)


def work(case):
    k = case["kind"]
    gb = {"f32": 44, "mixed": 20}  # G-buffer bytes per pixel
    geo = {"f32": 12, "mixed": 8}  # depth + normal
    rad = {"f32": 16, "mixed": 8}
    if k == "frame":
        px = case["w"] * case["h"]
        fl = _gather_flops(px, case["w"], case["dirs"], case["footprint"], case["steps"])
        fl += px * case["passes"] * (2 * case["radius"]) ** 2 * 18.0
        fmt = case["fmt"]
        by = geo[fmt] + rad[fmt] + 16 + (gb[fmt] - geo[fmt] - rad[fmt] if case["composite"] else 0)
        return {"bytes": px * by, "flops": fl}
    if k == "target":
        px = case["crop"] ** 2
        return {"bytes": px * (16 + 32), "flops": _gather_flops(px, case["w"], case["dirs"], 0, 0)}
    if k == "pyramid":
        px, t = case["w"] * case["h"], 1 if case["sampler"] == "trilinear" else 0
        up = sum(0.25 ** l for l in range(1, case["levels"]))
        return {"bytes": px * ((rad[case["fmt"]] + 4) + up * (2 * rad[case["fmt"]] + 4 * (1 + t))),
                "flops": px * up * (5 * 4 + 17 * 4 + (17 if t else 0))}
    if k == "bilateral":
        px = case["w"] * case["h"]
        return {"bytes": px * (32 + geo[case["fmt"]]), "flops": px * (2 * case["radius"]) ** 2 * 18.0}
    if k == "denoise":
        px = case["w"] * case["h"]
        return {"bytes": px * (32 + gb[case["fmt"]] - rad[case["fmt"]]), "flops": _unet_flops(px)}
    if k == "forward":
        px = case["n"] * case["w"] * case["h"]
        return {"bytes": px * 64, "flops": _unet_flops(px)}
    if k == "backward":
        px = case["n"] * case["w"] * case["h"]
        return {"bytes": px * 64, "flops": 3 * _unet_flops(px)}
    fl = by = 0
    for w, h in _views(case):
        fl += _gather_flops(w * h, w, 4, 256, 0)
        by += w * h * 32
    return {"bytes": by, "flops": fl}


def _views(case):
    return [tuple(int(x) for x in v.split("x")) for v in case["views"].split(",")]


# --------------------------------------------------------------------- inputs

def _camera(rng, w, h):
    """View and projection (column-major float32) of a 60 degree camera inside the room."""
    pos = rng.uniform([0.2, 0.45, 0.2], [0.8, 0.75, 0.8])
    hor, vert = rng.uniform(0, 2 * math.pi), rng.uniform(-0.35, -0.05)
    ch, sh, cv, sv = math.cos(hor), math.sin(hor), math.cos(vert), math.sin(vert)
    t = np.eye(4)
    t[:3, 3] = pos
    ry = np.array([[ch, 0, sh, 0], [0, 1, 0, 0], [-sh, 0, ch, 0], [0, 0, 0, 1]])
    rx = np.array([[1, 0, 0, 0], [0, cv, -sv, 0], [0, sv, cv, 0], [0, 0, 0, 1]])
    f, near, far = 1 / math.tan(math.pi / 6), 0.01, 10.0
    p = np.array([[f * h / w, 0, 0, 0], [0, f, 0, 0], [0, 0, -(far + near) / (far - near), -2 * far * near / (far - near)],
                  [0, 0, -1, 0]]) @ np.diag([1.0, -1.0, -1.0, 1.0])
    view = np.linalg.inv(t @ ry @ rx)
    return view.T.astype(np.float32).reshape(-1), p.T.astype(np.float32).reshape(-1)


def _unproject(inv, x, y):
    v = [inv[r, 0] * x + inv[r, 1] * y + (inv[r, 2] + inv[r, 3]) for r in range(4)]
    return torch.stack([v[0] / v[3], v[1] / v[3], v[2] / v[3]], -1)


def _mats(view, proj):
    v, p = (np.asarray(m, np.float64).reshape(4, 4).T for m in (view, proj))
    return np.linalg.inv(p @ v), np.linalg.inv(v)[:3, 3]


class _Room:
    """The unit cube seen from inside, with axis-aligned boxes and spheres."""

    def __init__(self, rng, boxes=32, spheres=8):
        size = rng.uniform(0.05, 0.3, (boxes, 3))
        lo = rng.uniform(0, 1, (boxes, 3)) * (1 - size) * [1, 0.4, 1]
        self.boxes = np.stack([lo, lo + size], 1)
        self.spheres = np.concatenate([rng.uniform(0.1, 0.9, (spheres, 3)) * [1, 0.5, 1],
                                       rng.uniform(0.05, 0.15, (spheres, 1))], 1)
        self.albedo = torch.tensor(rng.uniform(0.1, 0.9, (6 + boxes + spheres, 3)), dtype=torch.float32, device="cuda")
        d = rng.uniform([-0.6, 0.6, -0.6], [0.6, 1.0, 0.6])
        self.light = torch.tensor(d / np.linalg.norm(d), dtype=torch.float32, device="cuda")

    def cast(self, o, d, shell):
        """(distance, normal, object) of the first hit along o + t d; without the shell: whether anything is hit."""
        inv = 1 / torch.where(d.abs() < 1e-8, torch.full_like(d, 1e-8), d)
        far = torch.maximum(-o * inv, (1 - o) * inv)
        best, axis = far.min(-1)
        n = -torch.sign(d) * torch.nn.functional.one_hot(axis, 3)
        obj = axis * 2 + (torch.gather(d, -1, axis[..., None])[..., 0] > 0)
        hit = torch.zeros_like(best, dtype=torch.bool)
        for i, b in enumerate(torch.tensor(self.boxes, dtype=torch.float32, device="cuda")):
            t1, t2 = (b[0] - o) * inv, (b[1] - o) * inv
            near, ax = torch.minimum(t1, t2).max(-1)
            ok = (near < torch.maximum(t1, t2).min(-1)[0]) & (near > 1e-4) & (near < best)
            hit |= ok
            if shell:
                best = torch.where(ok, near, best)
                n = torch.where(ok[..., None], -torch.sign(d) * torch.nn.functional.one_hot(ax, 3), n)
                obj = torch.where(ok, 6 + i, obj)
        for i, s in enumerate(torch.tensor(self.spheres, dtype=torch.float32, device="cuda")):
            oc = o - s[:3]
            b = (oc * d).sum(-1)
            disc = b * b - ((oc * oc).sum(-1) - s[3] * s[3])
            t = -b - disc.clamp_min(0).sqrt()
            ok = (disc > 0) & (t > 1e-4) & (t < best)
            hit |= ok
            if shell:
                best = torch.where(ok, t, best)
                n = torch.where(ok[..., None], (oc + t[..., None] * d) / s[3], n)
                obj = torch.where(ok, 6 + len(self.boxes) + i, obj)
        return (best, n, obj) if shell else hit


def _scene(seed, w, h, fmt, part=0):
    """(G-buffer, view, proj) of a seeded room, in the storage formats of `fmt`."""
    rng = np.random.default_rng([int(seed), part])
    view, proj = _camera(rng, w, h)
    room = _Room(rng)
    inv, cam = _mats(view, proj)
    x = ((torch.arange(w, device="cuda", dtype=torch.float64) + 0.5) / w * 2 - 1).expand(h, w)
    y = ((torch.arange(h, device="cuda", dtype=torch.float64) + 0.5) / h * 2 - 1)[:, None].expand(h, w)
    cam = torch.tensor(cam, device="cuda")
    ray = torch.nn.functional.normalize(_unproject(inv, x, y) - cam, dim=-1).float()
    o = cam.float().expand(h, w, 3)
    depth, n, obj = room.cast(o, ray, True)
    p = o + ray * depth[..., None] + n * 1e-3
    lit = (n @ room.light).clamp_min(0) * ~room.cast(p, room.light.expand(h, w, 3), False)
    albedo = room.albedo[obj]
    rgba = lambda c: torch.cat([c, torch.ones_like(c[..., :1])], -1)  # noqa: E731
    e = n / n.abs().sum(-1, keepdim=True)
    fold = (1 - e[..., [1, 0]].abs()) * torch.where(e[..., :2] >= 0, 1.0, -1.0)
    octn = torch.where(e[..., 2:] < 0, fold, e[..., :2])
    f = lgx.GBUF_FORMATS[fmt]
    if fmt == "mixed":
        octn, al, ra = octn.half(), (rgba(albedo) * 255 + 0.5).to(torch.uint8), rgba(albedo * lit[..., None] * 3).half()
    else:
        al, ra = rgba(albedo), rgba(albedo * lit[..., None] * 3)
    im = lambda t, fm: dev.DImage(w, h, fm, tensor=t.contiguous())  # noqa: E731
    return dev.GBufferDev(im(depth, lgx.R32F), im(octn, f["normal"]), im(al, f["albedo"]), im(ra, f["radiance"])), view, proj


def _noise(seed, shape):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed) * 7919 + 17)
    return torch.randn(shape, device="cuda", generator=g)


def _noisy(seed, gb):
    """A few-direction irradiance of the scene: a smooth field of position and albedo under strong noise."""
    d = gb.depth.t[..., None]
    base = 0.15 + 0.1 * torch.cos(d * torch.tensor([2.0, 3.0, 4.0], device="cuda")) + 0.2 * gb.radiance.t[..., :3].float()
    c = base * (1 + 0.6 * _noise(seed, base.shape)).clamp_min(0)
    return dev.DImage(gb.w, gb.h, lgx.RGBA32F, tensor=torch.cat([c, torch.ones_like(d)], -1).contiguous()), base


def _albedo(gb):
    return gb.albedo.t[..., :3].float() / 255 if gb.albedo.fmt == lgx.RGBA8 else gb.albedo.t[..., :3]


def _records(case, seed):
    """Input records [n][h][w][12] and clean targets [n][h][w][4]: a frame's crops."""
    n, w, h = case["n"], case["w"], case["h"]
    gx = math.ceil(math.sqrt(n))
    gb, _, _ = _scene(seed, w * gx, h * gx, "mixed")
    noisy, base = _noisy(seed, gb)
    z = torch.zeros_like(base)
    rec = torch.cat([noisy.t[..., :3], gb.depth.t[..., None], gb.normal.t.float(), _albedo(gb), z], -1)
    cut = lambda t: (t.reshape(gx, h, gx, w, -1).permute(0, 2, 1, 3, 4).reshape(gx * gx, h, w, -1)[:n].contiguous())  # noqa: E731
    return cut(rec), cut(torch.cat([base, z[..., :1]], -1))


def _net(n, w, h, backward=False):
    net = dev.UNet(n, h, w)
    net.load(dn.WEIGHTS)
    net.autotune(n, h, w, backward=backward)
    return net


class _View:
    """An image inside a renderer or batch as a tensor (no copy); it keeps its owner, which frees the image, alive."""

    def __init__(self, im, owner):
        self.owner = owner
        self.__cuda_array_interface__ = {"shape": (im.h, im.w, 4), "typestr": "<f4", "data": (im.ptr, False), "version": 2,
                                         "strides": (im.pitch * 16, 16, 4)}


def _tensor(im, owner):
    t = torch.as_tensor(_View(im, owner), device="cuda")
    t.owner = owner  # the tensor's storage already refers to the view
    return t


def prepare(case, seed):
    k = case["kind"]
    s = dict(case=case)
    if k == "frame":
        s["gb"], s["view"], s["proj"] = _scene(seed, case["w"], case["h"], case["fmt"])
        s["r"] = dev.Renderer(case["w"], case["h"], case["dirs"], case["steps"], case["levels"],
                              lgx.SAMPLER_TRILINEAR if case["sampler"] == "trilinear" else lgx.SAMPLER_HIZ_POINT,
                              case["grid"], denoiser=lgx.DENOISER_BILATERAL if case["passes"] else lgx.DENOISER_NONE,
                              denoise_passes=case["passes"], denoise_radius=max(1, case["radius"]), kind=case["fmt"],
                              tile=case["tile"], composite=case["composite"], footprint_dirs=case["footprint"])
    elif k == "target":
        gb, s["view"], s["proj"] = _scene(seed, case["w"], case["h"], "mixed")
        s["gb"], s["pyr"] = gb, dev.PyramidDev(gb, case["levels"], lgx.SAMPLER_HIZ_POINT).build()
        s["g"] = dev.Gather(case["w"], case["h"], case["dirs"], 0, lgx.SAMPLER_HIZ_POINT,
                            precision=lgx.PREC_F64 if case["precision"] == "f64" else lgx.PREC_F32_ACC64)
        s["out"] = dev.DImage(case["w"], case["h"], lgx.RGBA64F)
        s["roi"] = _roi(case, seed)
    elif k == "pyramid":
        s["gb"], _, _ = _scene(seed, case["w"], case["h"], case["fmt"])
        tri = case["sampler"] == "trilinear"
        p = s["pyr"] = dev.PyramidDev(s["gb"], case["levels"], lgx.SAMPLER_TRILINEAR if tri else lgx.SAMPLER_HIZ_POINT)
        n = case["levels"]
        arr = lambda ims: (lgx.Image * len(ims))(*[d.desc for d in ims])  # noqa: E731
        s["mips"] = [(arr(p.rad), lgx.MIP_AVG), (arr(p.dep), lgx.MIP_AVG if tri else lgx.MIP_MAX)]
        s["blurs"] = [(arr(p.rad[1:]), arr(p.rad_b[1:]))] + ([(arr(p.dep[1:]), arr(p.dep_b[1:]))] if tri else [])
        s["radius"] = (C.c_int32 * (n - 1))(*([2] * (n - 1)))
    elif k == "bilateral":
        s["gb"], _, _ = _scene(seed, case["w"], case["h"], case["fmt"])
        s["in"], _ = _noisy(seed, s["gb"])
        s["out"] = dev.DImage(case["w"], case["h"], lgx.RGBA32F)
    elif k == "denoise":
        s["gb"], _, _ = _scene(seed, case["w"], case["h"], case["fmt"])
        s["in"], _ = _noisy(seed, s["gb"])
        s["out"] = dev.DImage(case["w"], case["h"], lgx.RGBA32F)
        s["net"] = _net(1, case["w"], case["h"])
    elif k in ("forward", "backward"):
        s["x"], s["t"] = _records(case, seed)
        s["net"] = _net(case["n"], case["w"], case["h"], backward=k == "backward")
        s["out"] = torch.empty_like(s["t"])
        s["loss"] = torch.zeros(1, device="cuda")
        if k == "backward":
            s["net"].set_loss(case["loss"])
    else:
        s["views"] = [_scene(seed, w, h, "mixed", i) for i, (w, h) in enumerate(_views(case))]
        s["batch"] = dev.Batch(s["views"], dirs=4, max_steps=0, levels=6, grid=8, footprint_dirs=256, tile=case["tile"])
        outs = []
        for i in range(len(s["views"])):
            im = lgx.Image()
            lgx.check(lgx.lib().lgx_batch_output(s["batch"].h, i, 0, C.byref(im)), "lgx_batch_output")
            outs.append(_tensor(im, s["batch"]))
        s["outs"] = outs
    return s


def _roi(case, seed):
    rng = np.random.default_rng([int(seed), 99])
    x0, y0 = (int(rng.integers(0, (e - case["crop"]) // 16 + 1)) * 16 for e in (case["w"], case["h"]))
    return (x0, y0, case["crop"], case["crop"])


def run(state):
    case = state["case"]
    k = case["kind"]
    if k == "frame":
        r = state["r"]
        r.render(state["gb"], state["view"], state["proj"])
        if "out" not in state:  # the renderer's output image stays where it is
            im = lgx.Image()
            name = b"final" if case["composite"] else b"denoised"
            lgx.check(lgx.lib().lgx_renderer_intermediate(r.h, name, 0, C.byref(im)), "lgx_renderer_intermediate")
            state["out"] = _tensor(im, r)
        return state["out"]
    if k == "target":
        x, y, w, h = state["roi"]
        state["g"](state["view"], state["proj"], state["gb"], state["pyr"], out=state["out"], roi=state["roi"])
        return state["out"].t[y:y + h, x:x + w]
    if k == "pyramid":
        lib, st, n = lgx.lib(), dev.stream_handle(), case["levels"]
        for lv, mode in state["mips"]:
            lgx.check(lib.lgx_mip_build(lv, n, mode, st), "lgx_mip_build")
        for a, b in state["blurs"]:
            lgx.check(lib.lgx_box_blur(a, b, state["radius"], n - 1, st), "lgx_box_blur")
        p = state["pyr"]
        out = dict(radiance=[i.t for i in p.rad[1:]], blurred=[i.t for i in p.rad_b[1:]], depth=[i.t for i in p.dep[1:]])
        if case["sampler"] == "trilinear":
            out["blurred_depth"] = [i.t for i in p.dep_b[1:]]
        return out
    if k == "bilateral":
        return dev.bilateral(state["in"], state["gb"], out=state["out"], radius=case["radius"]).t
    if k == "denoise":
        return state["net"].denoise(state["gb"], state["in"], out=state["out"]).t
    if k == "forward":
        return state["net"].forward(state["x"], out=state["out"])
    if k == "backward":
        state["net"].backward(state["x"], state["t"], state["loss"])
        return dict(loss=state["loss"], grads=state["net"].get(1)[0])
    state["batch"].run()
    return state["outs"]


# -------------------------------------------------------------- 64-bit results

def _mips(x, n, mode, store):
    """Pyramid of [h][w][c]: floor halving, each level rounded to its storage type."""
    out = [x]
    for _ in range(n - 1):
        h, w = out[-1].shape[0] // 2 * 2, out[-1].shape[1] // 2 * 2
        q = out[-1][:h, :w].reshape(h // 2, 2, w // 2, 2, -1)
        q = q.amax((1, 3)) if mode == "max" else q.sum((1, 3)) / 4
        out.append(q.to(store).double())
    return out


def _at(x, dy, dx):
    h, w = x.shape[:2]
    iy = (torch.arange(h, device=x.device) + dy).clamp(0, h - 1)
    ix = (torch.arange(w, device=x.device) + dx).clamp(0, w - 1)
    return x[iy][:, ix]


def _blur(x, store):
    s = sum(_at(x, dy, dx) for dx in range(-2, 2) for dy in range(-2, 2))
    return (s / 16).to(store).double()


def _pyramids(gb, n, sampler):
    store = gb.radiance.t.dtype
    rad = _mips(gb.radiance.t.double(), n, "avg", store)
    dep = _mips(gb.depth.t.double()[..., None], n, "max" if sampler == "hiz" else "avg", torch.float32)
    rb = rad[:1] + [_blur(x, store) for x in rad[1:]]
    db = dep if sampler == "hiz" else dep[:1] + [_blur(x, torch.float32) for x in dep[1:]]
    return rad, dep, rb, db


def _oct(e):
    z = 1 - e.abs().sum(-1, keepdim=True)
    fold = (1 - e[..., [1, 0]].abs()) * torch.where(e >= 0, 1.0, -1.0).double()
    v = torch.cat([torch.where(z < 0, fold, e), z], -1)
    return v / v.norm(dim=-1, keepdim=True)


def _hammersley(n):
    i = np.arange(n, dtype=np.uint64)
    rev = np.array([int(format(int(k), "032b")[::-1], 2) for k in i], np.float64)
    return i.astype(np.float32) / np.float32(n), rev.astype(np.float32) / np.float32(2.0 ** 32)


def _flat(levels):
    base = np.cumsum([0] + [x.shape[0] * x.shape[1] for x in levels[:-1]])
    t = lambda a: torch.tensor(a, device="cuda")  # noqa: E731
    return (torch.cat([x.reshape(-1, x.shape[-1]) for x in levels]), t(base), t([x.shape[1] for x in levels]),
            t([x.shape[0] for x in levels]))


def _point(fl, lod, sx, sy):
    data, base, lw, lh = fl
    l = lod.clamp(0, len(base) - 1).floor().long()
    w, h = lw[l], lh[l]
    ix, iy = (sx * w).floor().long(), (sy * h).floor().long()
    ix, iy = torch.minimum(ix.clamp_min(0), w - 1), torch.minimum(iy.clamp_min(0), h - 1)
    return data[base[l] + iy * w + ix]


def _bilinear(fl, l, sx, sy):
    data, base, lw, lh = fl
    w, h = lw[l], lh[l]
    u, v = sx * w - 0.5, sy * h - 0.5
    i, j = u.floor(), v.floor()
    a, b = (u - i)[..., None], (v - j)[..., None]
    cx = lambda k: torch.minimum(k.long().clamp_min(0), w - 1)  # noqa: E731
    cy = lambda k: torch.minimum(k.long().clamp_min(0), h - 1)  # noqa: E731
    p = lambda y, x: data[base[l] + cy(y) * w + cx(x)]  # noqa: E731
    return (p(j, i) * (1 - a) + p(j, i + 1) * a) * (1 - b) + (p(j + 1, i) * (1 - a) + p(j + 1, i + 1) * a) * b


def _trilinear(fl, lod, sx, sy):
    top = len(fl[1]) - 1
    d = lod.clamp(0, top)
    l = d.floor().long()
    f = (d - l)[..., None]
    return _bilinear(fl, l, sx, sy) * (1 - f) + _bilinear(fl, (l + 1).clamp_max(top), sx, sy) * f


def _gather(gb, view, proj, db, rb, dirs, steps, sampler, grid, footprint, roi=None):
    """The horizon gather (indirectLighting.frag:114-272) in double; [h][w][3] of the region."""
    W, H = gb.w, gb.h
    x0, y0, w, h = roi or (0, 0, W, H)
    y, x = (t.reshape(-1) for t in torch.meshgrid(torch.arange(y0, y0 + h, device="cuda"),
                                                  torch.arange(x0, x0 + w, device="cuda"), indexing="ij"))
    ang, lin = (torch.tensor(t.astype(np.float64), device="cuda") for t in _hammersley(grid * grid))
    k = x % grid + y % grid * grid
    ang, lin = ang[k], lin[k]
    inv, cam = _mats(view, proj)
    cam = torch.tensor(cam, device="cuda")
    at = lambda im: im.t[y0:y0 + h, x0:x0 + w].reshape(w * h, -1).double()  # noqa: E731
    rc, n = at(gb.depth), _oct(at(gb.normal))
    cx, cy = x + 0.5, y + 0.5
    ray = lambda px, py: torch.nn.functional.normalize(_unproject(inv, px / W * 2 - 1, py / H * 2 - 1) - cam, dim=-1)  # noqa: E731
    rayc = ray(cx.double(), cy.double())
    P = cam + rayc * rc
    eye = -rayc
    dot = lambda a, b: (a * b).sum(-1)  # noqa: E731
    near, Df = W / 1000.0, float(footprint or dirs)
    ratio = 2 * PI / Df + 1
    fd, fr = _flat(db), _flat(rb)
    sample = _trilinear if sampler == "trilinear" else _point
    en, total = dot(eye, n), torch.zeros(w * h, 3, dtype=torch.float64, device="cuda")
    chunk = max(1, min(dirs, (1 << 21) // (w * h)))
    for d0 in range(0, dirs, chunk):
        d = torch.arange(d0, min(dirs, d0 + chunk), device="cuda", dtype=torch.float64)[:, None]
        th = 2 * PI / dirs * (ang + d)
        dx, dy = th.cos(), th.sin()
        tan = torch.nn.functional.normalize(ray(cx + dx, cy + dy) - rayc, dim=-1)
        dn_ = torch.linalg.cross(-torch.linalg.cross(tan, eye.expand_as(tan)), n.expand_as(tan))
        mx = torch.atan2(dot(dn_, tan), dot(dn_, eye))
        tn = dot(tan, n)
        hc = lambda mn, mx: (0.25 * en * ((2 * mn).cos() - (2 * mx).cos()) +  # noqa: E731
                             0.25 * tn * (2 * mx - 2 * mn - (2 * mx).sin() + (2 * mn).sin()))
        L = (AMBIENT * hc(torch.zeros_like(mx), mx))[..., None].repeat(1, 1, 3)
        path = torch.minimum(torch.maximum(-cx / dx, (W - cx) / dx), torch.maximum(-cy / dy, (H - cy) / dy)).abs()
        iters = ((path / near).log() / math.log(ratio)).trunc() + 1
        if steps > 0:
            iters = iters.clamp_max(steps)
        for j in range(int(iters.max())):
            off = near * ratio ** (j + lin) + 1 - near
            sx, sy = (cx + dx * off) / W, (cy + dy * off) / H
            on = (j < iters) & (sx > 0) & (sx < 1) & (sy > 0) & (sy < 1)
            lod = ((2 * PI / Df * (off - 1) * 0.5).clamp_min(1e-30).log2() - 2).expand_as(sx)
            r = sample(fd, lod, sx, sy)
            dl = cam + ray(sx * W, sy * H) * r - P
            sh = torch.atan2(dot(tan, dl), dot(eye, dl))
            hit = on & (sh < mx)
            t = lambda s: (s / 0.1).clamp(0, 1)  # noqa: E731
            g = hc(sh, mx) * t(1 - sx) * t(sx) * t(1 - sy) * t(sy)
            L = torch.where(hit[..., None], L + (sample(fr, lod, sx, sy)[..., :3] - AMBIENT) * g[..., None], L)
            mx = torch.where(hit, sh, mx)
        total += (2 * L / dirs).sum(0)
    return total.reshape(h, w, 3)


def _bilateral(x, gb, r):
    d, n = gb.depth.t.double()[..., None], _oct(gb.normal.t.double())
    num, den = torch.zeros_like(x), torch.zeros_like(d)
    for dy in range(-r, r):
        for dx in range(-r, r):
            e = 10.5 * (_at(d, dy, dx) - d).abs() + 20.0 * (_at(n, dy, dx) - n).square().sum(-1, keepdim=True)
            wgt = (-e).exp()
            num += _at(x, dy, dx) * wgt
            den += wgt
    return num / (den + 1e-7)


def _rgba(c, a=None):
    return torch.cat([c, torch.ones_like(c[..., :1]) if a is None else a], -1)


def _params():
    """The committed network's layers [(W, b)] x 10 and head (W, b), from the safetensors file."""
    with open(dn.WEIGHTS, "rb") as f:
        head = json.loads(f.read(int.from_bytes(f.read(8), "little")))
        a, b = head["params"]["data_offsets"]
        f.seek(a, 1)
        flat = np.frombuffer(f.read(b - a), np.float32)
    return torch.tensor(flat.astype(np.float64), device="cuda")


def _conv(x, w, b):
    n, h, wd, ci = x.shape
    p = torch.nn.functional.pad(x, (0, 0, 1, 1, 1, 1))
    y = b
    for ky in range(3):
        for kx in range(3):
            y = y + p[:, ky:ky + h, kx:kx + wd].reshape(-1, ci) @ w[:, :, ky, kx].t().contiguous()
    return y.reshape(n, h, wd, -1).relu()


def _unet(flat, rec):
    ls, o = [], 0
    for ci, co in LAYERS:
        ls.append((flat[o:o + co * ci * 9].reshape(co, ci, 3, 3), flat[o + co * ci * 9:o + co * ci * 9 + co]))
        o += co * ci * 9 + co
    wh, bh = flat[o:o + 96].reshape(3, 32), flat[o + 96:o + 99]
    pool = lambda x: x.reshape(x.shape[0], x.shape[1] // 2, 2, x.shape[2] // 2, 2, -1).mean((2, 4))  # noqa: E731
    up = lambda x: x.repeat_interleave(2, 1).repeat_interleave(2, 2)  # noqa: E731
    e1 = _conv(_conv(rec[..., :9], *ls[0]), *ls[1])
    e2 = _conv(_conv(pool(e1), *ls[2]), *ls[3])
    b = _conv(_conv(pool(e2), *ls[4]), *ls[5])
    d2 = _conv(_conv(torch.cat([up(b), e2], -1), *ls[6]), *ls[7])
    d1 = _conv(_conv(torch.cat([up(d2), e1], -1), *ls[8]), *ls[9])
    return rec[..., :3] + (d1.reshape(-1, 32) @ wh.t() + bh).reshape(rec[..., :3].shape)


def exact(case, seed):
    k = case["kind"]
    with torch.no_grad():
        if k == "frame":
            gb, view, proj = _scene(seed, case["w"], case["h"], case["fmt"])
            _, _, rb, db = _pyramids(gb, case["levels"], case["sampler"])
            x = _gather(gb, view, proj, db, rb, case["dirs"], case["steps"], case["sampler"], case["grid"], case["footprint"])
            for _ in range(case["passes"]):
                x = _bilateral(x, gb, case["radius"])
            if not case["composite"]:
                return _rgba(x)
            al = gb.albedo.t.double() / (255 if gb.albedo.fmt == lgx.RGBA8 else 1)
            return gb.radiance.t.double() + _rgba(x) * al
        if k == "target":
            gb, view, proj = _scene(seed, case["w"], case["h"], "mixed")
            _, _, rb, db = _pyramids(gb, case["levels"], "hiz")
            return _rgba(_gather(gb, view, proj, db, rb, case["dirs"], 0, "hiz", 4, 0, _roi(case, seed)))
        if k == "pyramid":
            gb, _, _ = _scene(seed, case["w"], case["h"], case["fmt"])
            rad, dep, rb, db = _pyramids(gb, case["levels"], case["sampler"])
            out = dict(radiance=rad[1:], blurred=rb[1:], depth=[x[..., 0] for x in dep[1:]])
            if case["sampler"] == "trilinear":
                out["blurred_depth"] = [x[..., 0] for x in db[1:]]
            return out
        if k in ("bilateral", "denoise"):
            gb, _, _ = _scene(seed, case["w"], case["h"], case["fmt"])
            x = _noisy(seed, gb)[0].t.double()[..., :3]
            if k == "bilateral":
                return _rgba(_bilateral(x, gb, case["radius"]))
            al = gb.albedo.t.double()[..., :3] / (255 if gb.albedo.fmt == lgx.RGBA8 else 1)
            rec = torch.cat([x, gb.depth.t.double()[..., None], gb.normal.t.double(), al], -1)
            return _rgba(_unet(_params(), rec[None])[0])
        if k == "forward":
            return _rgba(_unet(_params(), _records(case, seed)[0].double()))
        if k == "batch":
            out = []
            for i, (w, h) in enumerate(_views(case)):
                gb, view, proj = _scene(seed, w, h, "mixed", i)
                _, _, rb, db = _pyramids(gb, 6, "hiz")
                out.append(_rgba(_gather(gb, view, proj, db, rb, 4, 0, "hiz", 8, 256)))
            return out
    rec, tgt = (t.double() for t in _records(case, seed))
    flat = _params().requires_grad_()
    diff = _unet(flat, rec) - tgt[..., :3]
    loss = diff.abs().mean() if case["loss"] == "l1" else diff.square().mean()
    loss.backward()
    return dict(loss=loss.detach().reshape(1), grads=flat.grad)
