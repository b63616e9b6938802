"""FP64 sums keep the shader's own end of the march (indirectLighting.frag:212
and the screen test), FP32 sums end at an offset limit that may differ from it
by a step within rounding.  Both ends are restated here in float32 for a row of
a 1080p frame of 256 directions that holds such places: per pixel and
direction the rule's count (the logarithm on the device, as the kernel has
it) and the limit's, the far borders' 2^-20 included.  With bright borders,
where such a step is, a pixel may differ between the two precisions only where
the counts do, and some do: elsewhere the steps are the same and the sums
within the gather's bar of 1e-4."""
import ctypes as C

import numpy as np
import pytest

torch = pytest.importorskip("torch")

from legitengine_amd import lgx  # noqa: E402

pytestmark = pytest.mark.gpu

W, H, D, ROW = 1920, 1080, 256, 490
F = np.float32
PI = F(3.1415)


def libm(name, *args):
    fn = getattr(C.CDLL("libm.so.6"), name)
    fn.restype, fn.argtypes = C.c_float, [C.c_float] * len(args)
    return F(fn(*[float(a) for a in args]))


def tables(k):
    """Directions and offsets of pattern index k, by the host's own functions."""
    ang, lin = F(k) / F(16), F(int(f"{k:04b}"[::-1], 2)) / F(16)  # Hammersley of 16
    near, ratio = F(W) / F(1000), F(2) * PI / F(D) + F(1)
    step = F(2) * PI / F(D)
    dirs = [(libm("cosf", a), libm("sinf", a)) for a in (step * ang + step * F(d) for d in range(D))]
    n = int(libm("logf", np.sqrt(F(W) * F(W) + F(H) * F(H)) / near) / libm("logf", ratio)) + 2
    off = [near * libm("powf", ratio, F(j) + lin) + F(1) - near for j in range(n)]
    return np.array(dirs, F), np.array(off, F), near, ratio


def ends(k, xs):
    """[pixel, direction]: the steps that the rule and the limit take."""
    dirs, off, near, ratio = tables(k)
    t = lambda a: torch.from_numpy(np.ascontiguousarray(a, F)).cuda()  # noqa: E731
    dx, dy, o = t(dirs[:, 0]), t(dirs[:, 1]), t(off)
    idx, idy = t(F(1) / dirs[:, 0]), t(F(1) / dirs[:, 1])
    cx, cy = t(xs + F(0.5))[:, None], F(ROW) + F(0.5)
    path = torch.minimum(torch.maximum((0 - cx) * idx, (W - cx) * idx),
                         torch.maximum(t(F(0) - cy) * idy, t(F(H) - cy) * idy)).abs()
    log_ratio = libm("logf", ratio)
    # (a division by a scalar is a product with its reciprocal in torch: divide by tensors)
    iters = (torch.log(path / torch.full_like(path, float(near))) / torch.full_like(path, float(log_ratio))).int() + 1
    iters = iters.clamp(max=len(off))
    qx = cx[..., None] + dx[:, None] * o
    qy = (dy[:, None] * o + float(cy)).expand_as(qx)
    seen = ((qx > 0) & (qx < W) & (qy > 0) & (qy < H)).int().cumprod(-1).sum(-1)
    rlin = (F(off[0]) - F(1) + near) / near
    grown = (path.double() * float(rlin) + float(F(1) - near)).float()  # (one rounding, as the fused operation)
    lim = torch.where(path >= float(near), grown, torch.where(path > float(near / ratio), o[1], torch.zeros_like(path)))
    lim = torch.minimum(lim, path)
    far = float(F(1) - F(2.0 ** -20))
    lim = torch.where(dx > 0, torch.minimum(lim, (W * far - cx) * idx), lim)
    lim = torch.where(dy > 0, torch.minimum(lim, (t(F(H) * F(far)) - float(cy)) * idy), lim)
    taken = (o[None, None] < lim[..., None]).sum(-1)
    return torch.minimum(iters, seen).cpu().numpy(), taken.cpu().numpy()


def test_fp64_sums_end_by_the_rule():
    from legitengine_amd import device as dev
    dev.require_device()
    sc = lgx.make_scene(3, 8, 2)
    view, proj = lgx.scene_matrices(sc, W, H)
    g = dev.GBufferDev.from_host(lgx.render_gbuffer_cpu(sc, W, H, "f32"))
    pyr = dev.PyramidDev(g, 5, lgx.SAMPLER_HIZ_POINT).build()
    for level in pyr.rad_b:
        for edge in (level.t[0], level.t[-1], level.t[:, 0], level.t[:, -1]):
            edge.fill_(1e6)
    out = {}
    for p in (lgx.PREC_F32, lgx.PREC_F32_ACC64):
        out[p] = dev.Gather(W, H, D, 0, lgx.SAMPLER_HIZ_POINT, precision=p)(view, proj, g, pyr, roi=(0, ROW, W, 1))
    torch.cuda.synchronize()
    a, b = (out[p].numpy()[ROW, :, :3].astype(np.float64) for p in (lgx.PREC_F32_ACC64, lgx.PREC_F32))
    differ = np.abs(a - b).max(-1) > 1e-4 * np.abs(a).max(-1)
    places = np.zeros(W, bool)
    for kx in range(4):
        xs = np.arange(kx, W, 4).astype(F)
        rule, limit = ends(kx + 4 * (ROW % 4), xs)
        places[kx::4] = (rule < limit).any(1) | (rule > limit).any(1)
    assert not (differ & ~places).any(), np.argwhere(differ & ~places)[:8]
    assert int(differ.sum()) > 10, (int(differ.sum()), int(places.sum()))
