"""The trilinear gather where a tap pair straddles a border texel and a
neighbour of another magnitude: the outermost half texel of a level (2^l / 2
pixels of the frame) takes the border's texel alone, whatever stands beside
it (a far-plane or an infinite depth), as the oracle's clamped taps do.  The
gather's existing bar, 1e-4 relative L2."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

from legitengine_amd import lgx  # noqa: E402
from oracle import binding as orc  # noqa: E402

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", [lgx.PREC_F32, lgx.PREC_F64])
@pytest.mark.parametrize("value", [1e8, np.inf])
@pytest.mark.parametrize("w,h,n", [(64, 36, 6), (97, 61, 5), (16, 16, 5)])
def test_border_texel_beside_a_far_one(w, h, n, value, precision):
    from legitengine_amd import device as dev
    dev.require_device()
    sc = lgx.make_scene(3, 8, 2)
    view, proj = lgx.scene_matrices(sc, w, h)
    gb = lgx.render_gbuffer_cpu(sc, w, h, "f32")
    g = dev.GBufferDev.from_host(gb)
    pyr = dev.PyramidDev(g, n, lgx.SAMPLER_TRILINEAR).build()
    torch.cuda.synchronize()
    changed = 0
    for d in pyr.dep_b[1:]:  # one texel inside every border of two or more
        a = d.numpy()
        for at in [(slice(None), 1), (slice(None), -2), (1, slice(None)), (-2, slice(None))]:
            if a.shape[0] > 1 and a.shape[1] > 1:
                edge = (a[:, 0].copy(), a[:, -1].copy(), a[0].copy(), a[-1].copy())
                a[at] = value
                a[:, 0], a[:, -1], a[0], a[-1] = edge
                changed += 1
        d.t.copy_(torch.from_numpy(a))
    assert changed
    out = dev.Gather(w, h, 8, 0, lgx.SAMPLER_TRILINEAR, precision=precision)(view, proj, g, pyr)
    torch.cuda.synchronize()
    ref = orc.gather(view, proj, gb["depth"], orc.widen(gb["normal"]), [d.numpy() for d in pyr.dep_b],
                     [orc.widen(r.numpy()) for r in pyr.rad_b], 8, 0, lgx.SAMPLER_TRILINEAR,
                     precision="f32" if precision == lgx.PREC_F32 else "f64")
    assert np.isfinite(ref).all() and np.isfinite(out.numpy()).all()
    assert orc.rel_l2(out.numpy(), ref) <= 1e-4
