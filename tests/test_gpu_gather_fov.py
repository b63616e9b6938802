"""Narrow fields of view: a pixel's angle is so small that rounding the slice's
tangent, the difference of two unit rays, decides signs of the horizon test,
and the shader's own float arithmetic is far from the exact image (24 % at 2
degrees and 640 pixels).  The kernel follows that arithmetic: at most a tenth
of that distance from the FP32 oracle, for both samplers and both sums."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

from legitengine_amd import lgx  # noqa: E402
from oracle import binding as orc  # noqa: E402

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", [lgx.PREC_F32, lgx.PREC_F32_ACC64])
@pytest.mark.parametrize("sampler", [lgx.SAMPLER_HIZ_POINT, lgx.SAMPLER_TRILINEAR])
def test_narrow_field_of_view(sampler, precision):
    from legitengine_amd import device as dev
    dev.require_device()
    w, h = 640, 360
    sc = lgx.make_scene(3, 8, 2)
    view, proj = lgx.scene_matrices(sc, w, h)
    proj = list(proj)
    for i in (0, 5):
        proj[i] *= 32  # 60 to 2 degrees
    gb = lgx.render_gbuffer_cpu(sc, w, h, "f32")
    g = dev.GBufferDev.from_host(gb)
    pyr = dev.PyramidDev(g, 5, sampler).build()
    out = dev.Gather(w, h, 8, 0, sampler, precision=precision)(view, proj, g, pyr)
    torch.cuda.synchronize()
    dep = [d.numpy() for d in pyr.dep_b]
    rad = [orc.widen(r.numpy()) for r in pyr.rad_b]
    args = (view, proj, gb["depth"], orc.widen(gb["normal"]), dep, rad, 8, 0, sampler)
    ref, exact = orc.gather(*args)[..., :3].astype(np.float64), orc.gather(*args, precision="f64")[..., :3]
    own = np.linalg.norm(ref - exact)
    assert own > 0.1 * np.linalg.norm(exact)
    assert np.linalg.norm(out.numpy()[..., :3].astype(np.float64) - ref) <= 0.1 * own
