"""The bilateral's output tiles: one output a thread (32 x 8 pixels) and two
(32 x 16, from 2 Mpixel on), at extents around the tiles' edges and every
radius, against the FP32 oracle (its existing bar, 1e-5 relative L2)."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

from legitengine_amd import lgx  # noqa: E402
from oracle import binding as orc  # noqa: E402

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("w,h,radius,kind", [(1, 1, 1, "f32"), (33, 9, 3, "mixed"), (31, 7, 7, "f32"), (32, 8, 6, "mixed"),
                                             (65, 17, 8, "mixed"), (2049, 1025, 1, "mixed"), (2048, 1024, 4, "f32")])
def test_bilateral_tile_edges(w, h, radius, kind):
    from legitengine_amd import device as dev
    dev.require_device()
    sc = lgx.make_scene(9, 8, 2)
    gb = lgx.render_gbuffer_cpu(sc, w, h, kind)
    g = dev.GBufferDev.from_host(gb)
    inp = np.random.default_rng(w + radius).random((h, w, 4), dtype=np.float32)
    out = dev.DImage(w, h, lgx.RGBA32F)
    out.t.fill_(-1.0)
    dev.bilateral(dev.DImage.from_numpy(inp, lgx.RGBA32F), g, out=out, radius=radius)
    torch.cuda.synchronize()
    ref = orc.bilateral(inp, gb["depth"], orc.widen(gb["normal"]), radius)
    assert orc.rel_l2(out.numpy(), ref) <= 1e-5
    assert (out.numpy()[..., 3] == 1.0).all()
