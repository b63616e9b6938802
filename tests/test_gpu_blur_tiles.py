"""The pyramids' pre-blur (r = 2, tiles of 64 x 16) at extents around its
tiles' edges, several images and formats per launch, bit for bit against the
oracle; and a launch of mixed radii, which takes the general kernel."""
import ctypes as C

import numpy as np
import pytest

torch = pytest.importorskip("torch")

from legitengine_amd import lgx  # noqa: E402
from oracle import binding as orc  # noqa: E402

pytestmark = pytest.mark.gpu

SIZES = [(1, 1), (2, 3), (63, 4), (64, 16), (65, 17), (130, 33), (5, 70)]


@pytest.mark.parametrize("radii", [[2] * 7, [2, 1, 2, 3, 2, 2, 0]])
@pytest.mark.parametrize("fmt,ch,half", [(lgx.R32F, 1, False), (lgx.RG32F, 2, False), (lgx.RGBA16F, 4, True),
                                         (lgx.RGBA32F, 4, False)])
def test_blur_tile_edges(radii, fmt, ch, half):
    from legitengine_amd import device as dev
    dev.require_device()
    rng = np.random.default_rng(ch)
    arrs = [rng.standard_normal((h, w, ch)).astype(np.float16 if half else np.float32) for w, h in SIZES]
    src = [dev.DImage.from_numpy(a, fmt) for a in arrs]
    dst = [dev.DImage(w, h, fmt) for w, h in SIZES]
    n = len(SIZES)
    lgx.check(lgx.lib().lgx_box_blur((lgx.Image * n)(*[i.desc for i in src]), (lgx.Image * n)(*[i.desc for i in dst]),
                                     (C.c_int32 * n)(*radii), n, dev.stream_handle()))
    torch.cuda.synchronize()
    for a, d, r in zip(arrs, dst, radii):
        ref = orc.box_blur(a.astype(np.float32), r, round_fp16=half)
        assert d.numpy().reshape(a.shape).astype(np.float32).tobytes() == ref.reshape(a.shape).astype(np.float32).tobytes()
