"""The gather forms directions only, so the unit of length is free: a scene,
its camera and its far plane times a power of two give the same image, far
beyond the magnitudes whose squares the short roots cover; and a radial
distance of next to nothing (a marker of the background) at a camera in the
origin has a finite pixel, as the oracle's IEEE arithmetic gives."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

from legitengine_amd import lgx  # noqa: E402
from oracle import binding as orc  # noqa: E402

pytestmark = pytest.mark.gpu

W, H, LEVELS = 96, 54, 5


def setup():
    from legitengine_amd import device as dev
    dev.require_device()
    sc = lgx.make_scene(5, 8, 2)
    view, proj = lgx.scene_matrices(sc, W, H)
    return dev, list(view), list(proj), lgx.render_gbuffer_cpu(sc, W, H, "f32")


def gather(dev, view, proj, gb, sampler):
    g = dev.GBufferDev.from_host(gb)
    pyr = dev.PyramidDev(g, LEVELS, sampler).build()
    out = dev.Gather(W, H, 8, 0, sampler)(view, proj, g, pyr)
    torch.cuda.synchronize()
    return out.numpy()


HIZ, TRI = lgx.SAMPLER_HIZ_POINT, lgx.SAMPLER_TRILINEAR
# (the Hi-Z path's hits take the hardware's reciprocal of a square, which is not subnormal from depths of 1e-18 on)


@pytest.mark.parametrize("sampler,exponent", [(s, e) for s in (HIZ, TRI) for e in (-45, -20, 20, 50)] + [(TRI, -60)])
def test_unit_of_length(sampler, exponent):
    """Powers of two scale every operation exactly: 1e-6 is far above what may
    differ (the host's inverse matrices) and far below a wrong direction."""
    dev, view, proj, gb = setup()
    ref = gather(dev, view, proj, gb, sampler)
    s = 2.0 ** exponent
    gb["depth"] = (gb["depth"] * np.float32(s)).astype(np.float32)
    for i in (12, 13, 14):
        view[i] *= s
    proj[14] *= s  # 2 far near / (near - far)
    out = gather(dev, view, proj, gb, sampler)
    assert np.isfinite(out).all()
    assert orc.rel_l2(out, ref) <= 1e-6


@pytest.mark.parametrize("sampler,marker", [(HIZ, 1e-15), (TRI, 1e-15), (TRI, 1e-20), (HIZ, -1.0), (TRI, -1.0)])
def test_distances_of_next_to_nothing(sampler, marker):
    dev, view, proj, gb = setup()
    for i in (12, 13, 14):
        view[i] = 0.0
    rng = np.random.default_rng(7)
    gb["depth"] = np.where(rng.random((H, W)) < 0.1, np.float32(marker), gb["depth"]).astype(np.float32)
    out = gather(dev, view, proj, gb, sampler)
    g = dev.GBufferDev.from_host(gb)
    pyr = dev.PyramidDev(g, LEVELS, sampler).build()
    torch.cuda.synchronize()
    ref = orc.gather(view, proj, gb["depth"], orc.widen(gb["normal"]), [d.numpy() for d in pyr.dep_b],
                     [orc.widen(r.numpy()) for r in pyr.rad_b], 8, 0, sampler)
    assert np.isfinite(ref).all()
    assert np.isfinite(out).all()
    assert orc.rel_l2(out, ref) <= 1e-4
