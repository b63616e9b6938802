"""The bilateral over the depths, sharpnesses and irradiances that it accepts
outside a room of unit size, against the FP32 oracle.  The weights depend on
differences of depth and normal; both sides subtract the same FP32 values, so
their distance from the camera and the size of the sharpness leave the
filter's existing bar (1e-5 relative L2) as it is: what remains are roundings
of the exponent relative to itself (2^-22 of at most 20 before the weight is
below 2e-9) and of the sums."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

from legitengine_amd import lgx  # noqa: E402
from oracle import binding as orc  # noqa: E402

pytestmark = pytest.mark.gpu


def run(w, h, radius, depth=None, ds=10.5, ns=20.0, irradiance=None):
    from legitengine_amd import device as dev
    dev.require_device()
    gb = lgx.render_gbuffer_cpu(lgx.make_scene(9, 8, 2), w, h, "f32")
    rng = np.random.default_rng(w + radius)
    if depth is not None:
        gb["depth"] = depth(gb["depth"], rng).astype(np.float32)
    inp = rng.random((h, w, 4), dtype=np.float32)
    if irradiance is not None:
        inp = irradiance(inp)
    out = dev.bilateral(dev.DImage.from_numpy(inp, lgx.RGBA32F), dev.GBufferDev.from_host(gb), radius=radius, ds=ds,
                        ns=ns)
    torch.cuda.synchronize()
    return out.numpy(), orc.bilateral(inp, gb["depth"], orc.widen(gb["normal"]), radius, ds, ns)


SIZES = [(67, 45, 4), (2048, 1024, 2)]  # one output a thread, two


@pytest.mark.parametrize("w,h,radius", SIZES)
@pytest.mark.parametrize("far,ds", [(1e3, 10.5), (1e4, 10.5), (1e3, 100.0)])
def test_depths_far_from_the_camera(w, h, radius, far, ds):
    out, ref = run(w, h, radius, lambda d, rng: far + d * 2.0 / ds + rng.random(d.shape) / ds, ds=ds)
    assert orc.rel_l2(out, ref) <= 1e-5


@pytest.mark.parametrize("w,h,radius", SIZES)
def test_background_at_the_largest_float(w, h, radius):
    big = float(np.finfo(np.float32).max)
    out, ref = run(w, h, radius, lambda d, rng: np.where(rng.random(d.shape) < 0.3, big, d))
    assert np.isfinite(out).all()
    assert orc.rel_l2(out, ref) <= 1e-5


@pytest.mark.parametrize("w,h,radius", SIZES)
def test_negative_depth_sharpness(w, h, radius):
    out, ref = run(w, h, radius, ds=-1.5)
    assert orc.rel_l2(out, ref) <= 1e-5


@pytest.mark.parametrize("w,h,radius", SIZES)
@pytest.mark.parametrize("ns", [-0.5, 0.0, 1e4, 1e6])
def test_normal_sharpness(w, h, radius, ns):
    out, ref = run(w, h, radius, ns=ns)
    assert np.isfinite(out).all()
    assert orc.rel_l2(out, ref) <= 1e-5


@pytest.mark.parametrize("w,h,radius", SIZES)
def test_infinite_irradiance(w, h, radius):
    """Taps of +inf and -inf: sums of one sign stay infinite, mixed ones are
    NaN, as the oracle's."""
    def spots(a):
        a[5:h // 4, 3, 0] = np.inf
        a[7, 9:w // 3, 1] = -np.inf
        a[h // 2, w // 2, 2] = np.inf
        a[h // 2 + 1, w // 2 + 1, 2] = -np.inf
        return a
    out, ref = run(w, h, radius, ns=5.0, irradiance=spots)  # (no weight so small that it may be flushed to 0)
    assert np.isinf(ref).any() and np.isnan(ref).any()
    assert np.array_equal(np.isnan(out), np.isnan(ref))
    assert np.array_equal(out[np.isinf(ref)], ref[np.isinf(ref)])
    f = np.isfinite(ref)
    assert np.isfinite(out[f]).all()
    assert np.linalg.norm((out[f] - ref[f]).astype(np.float64)) <= 1e-5 * np.linalg.norm(ref[f].astype(np.float64))


@pytest.mark.parametrize("w,h,radius", SIZES)
def test_normals_of_any_length(w, h, radius):
    """Encoded normals far outside the square: a length whose square overflows
    divides to zero, as in the oracle."""
    from legitengine_amd import device as dev
    dev.require_device()
    gb = lgx.render_gbuffer_cpu(lgx.make_scene(9, 8, 2), w, h, "f32")
    gb["normal"][3:h // 3, ::5] *= np.float32(1e21)
    gb["normal"][h // 2:, ::7] *= np.float32(1e6)
    inp = np.random.default_rng(w).random((h, w, 4), dtype=np.float32)
    out = dev.bilateral(dev.DImage.from_numpy(inp, lgx.RGBA32F), dev.GBufferDev.from_host(gb), radius=radius)
    torch.cuda.synchronize()
    ref = orc.bilateral(inp, gb["depth"], orc.widen(gb["normal"]), radius)
    assert np.isfinite(ref).all()
    assert orc.rel_l2(out.numpy(), ref) <= 1e-5
