"""The gather's direction split: the waves of a workgroup share the directions
of 64 pixels and their shares are added in direction order, so the result is
the step-counting kernel's (one wave per pixel) bit for bit, whatever the
split; and within the gather's bar (1e-4 relative L2) of the FP32 oracle."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

from legitengine_amd import lgx  # noqa: E402
from oracle import binding as orc  # noqa: E402

pytestmark = pytest.mark.gpu


# (extent, region, pattern, directions): fewer directions than waves, counts
# that no wave count divides, one more and one less than a round of 16 (and
# several rounds), tiles with a single pixel, extents the pattern does not
# divide; 1024 x 1040 x 4 directions crosses to the two-wave launch
CASES = [((5, 3), None, 4, 1), ((33, 18), None, 4, 2), ((64, 48), None, 4, 3), ((130, 70), None, (4, 16), 5),
         ((96, 64), (37, 11, 1, 1), 4, 15), ((96, 64), None, 8, 16), ((67, 45), (1, 2, 40, 33), 4, 17),
         ((64, 64), None, 4, 33), ((40, 24), None, 2, 256), ((1024, 1040), None, 4, 4)]


@pytest.mark.parametrize("sampler", [lgx.SAMPLER_HIZ_POINT, lgx.SAMPLER_TRILINEAR])
@pytest.mark.parametrize("extent,roi,grid,dirs", CASES)
def test_split_matches_one_wave_and_oracle(extent, roi, grid, dirs, sampler):
    from legitengine_amd import device as dev
    dev.require_device()
    w, h = extent
    levels = 1 if min(extent) < 16 else 4
    sc = lgx.make_scene(5, 8, 2)
    view, proj = lgx.scene_matrices(sc, w, h)
    gb = lgx.render_gbuffer_cpu(sc, w, h, "f32")
    g = dev.GBufferDev.from_host(gb)
    pyr = dev.PyramidDev(g, levels, sampler).build()
    x, y, rw, rh = roi or (0, 0, w, h)
    for prec in (lgx.PREC_F32, lgx.PREC_F32_ACC64):
        ga = dev.Gather(w, h, dirs, 64, sampler, grid=grid, precision=prec)
        a, b = (dev.DImage(w, h, ga.out_fmt) for _ in range(2))
        a.t.fill_(-3.0)
        b.t.fill_(-3.0)
        counts = torch.zeros((h, w), dtype=torch.int32, device="cuda")
        ga(view, proj, g, pyr, out=a, roi=roi)
        ga(view, proj, g, pyr, out=b, roi=roi, step_counts=counts)
        torch.cuda.synchronize()
        assert a.numpy().tobytes() == b.numpy().tobytes()
        outside = np.ones((h, w), bool)
        outside[y:y + rh, x:x + rw] = False
        assert (a.numpy()[outside] == -3.0).all()
        if prec == lgx.PREC_F32 and w * h <= 10000:
            dep, rad = [d.numpy() for d in pyr.dep_b], [r.numpy() for r in pyr.rad_b]
            ref = orc.gather(view, proj, gb["depth"], orc.widen(gb["normal"]), dep, rad, dirs, 64, sampler, grid=grid)
            assert orc.rel_l2(a.numpy()[y:y + rh, x:x + rw], ref[y:y + rh, x:x + rw]) <= 1e-4


@pytest.mark.parametrize("kind", ["f32", "mixed"])
@pytest.mark.parametrize("w,h,levels", [(9, 40, 4), (40, 9, 4), (4, 70, 3), (37, 21, 5)])
def test_trilinear_narrow_levels(w, h, levels, kind):
    """Trilinear taps come in pairs of neighbouring texels: levels one texel
    wide or high, odd extents and every border, against the FP32 oracle (the
    gather's bar)."""
    from legitengine_amd import device as dev
    dev.require_device()
    sc = lgx.make_scene(6, 8, 2)
    view, proj = lgx.scene_matrices(sc, w, h)
    gb = lgx.render_gbuffer_cpu(sc, w, h, kind)
    g = dev.GBufferDev.from_host(gb)
    pyr = dev.PyramidDev(g, levels, lgx.SAMPLER_TRILINEAR).build()
    out = dev.Gather(w, h, 4, 0, lgx.SAMPLER_TRILINEAR)(view, proj, g, pyr)
    torch.cuda.synchronize()
    dep, rad = [d.numpy() for d in pyr.dep_b], [orc.widen(r.numpy()) for r in pyr.rad_b]
    ref = orc.gather(view, proj, gb["depth"], orc.widen(gb["normal"]), dep, rad, 4, 0, lgx.SAMPLER_TRILINEAR)
    assert orc.rel_l2(out.numpy(), ref) <= 1e-4
