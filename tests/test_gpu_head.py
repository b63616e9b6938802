"""The network's 1x1 head in the last convolution's epilogue, by itself: with
weights under which every layer hands its first channels on unchanged, the
last activations are the input's channels rounded to BF16 (a different value
in every pixel and channel), and out = in + b + W act, added channel by
channel in FP32, has the same bits on the CPU.  Extents below, at and past
the tile of 8 x 32 pixels, several images, workgroups that walk several tiles;
the noisy image and the output with rows longer than the image, whose padding
is neither read into it nor written."""
import ctypes as C

import numpy as np
import pytest

torch = pytest.importorskip("torch")

from legitengine_amd import lgx  # noqa: E402
from oracle import unet_ref as U  # noqa: E402

pytestmark = pytest.mark.gpu

SIZES = [(1, 4, 4), (1, 8, 32), (2, 20, 44), (3, 36, 68), (1, 520, 1000)]


@pytest.fixture(scope="module")
def dev():
    from legitengine_amd import device
    device.require_device()
    return device


def passing_network(dev, n, h, w):
    """Layers 0, 1, 8 and 9 hand channel c % 9 of the input on as their channel c (the centre tap of each; layer
    8 through the skip, which follows 64 channels from below); the head has random weights."""
    layers = [(np.zeros((co, ci, 3, 3)), np.zeros(co)) for ci, co in U.LAYERS]
    for c in range(32):
        layers[0][0][c, c % 9, 1, 1] = 1.0
        layers[1][0][c, c, 1, 1] = 1.0
        layers[8][0][c, 64 + c, 1, 1] = 1.0
        layers[9][0][c, c, 1, 1] = 1.0
    rng = np.random.default_rng(5)
    wh, bh = rng.standard_normal((3, 32)), rng.standard_normal(3)
    flat = U.pack(layers, wh, bh).astype(np.float32)
    net = dev.UNet(n, h, w, seed=1)
    net.set(0, flat)
    return net, wh.astype(np.float32), bh.astype(np.float32)


def head(x9, wh, bh):
    """In FP32, in the kernel's order: input + bias, then channel by channel."""
    act = torch.from_numpy(np.ascontiguousarray(x9)).to(torch.bfloat16).to(torch.float32).numpy()
    act = np.maximum(act, np.float32(0))
    out = np.empty(x9.shape[:-1] + (4,), np.float32)
    for k in range(3):
        o = x9[..., k] + bh[k]
        for i in range(32):
            o = o + wh[k, i] * act[..., i % 9]
        out[..., k] = o
    out[..., 3] = 1.0
    return out


@pytest.mark.parametrize("n,h,w", SIZES)
def test_forward(dev, n, h, w):
    net, wh, bh = passing_network(dev, n, h, w)
    x = np.random.default_rng(h).standard_normal((n, h, w, 12)).astype(np.float32)
    out = net.forward(torch.from_numpy(x).cuda()).cpu().numpy()
    assert out.tobytes() == head(x[..., :9], wh, bh).tobytes()


@pytest.mark.parametrize("pad", [0, 5])
@pytest.mark.parametrize("h,w", [(h, w) for n, h, w in SIZES if n == 1])
def test_denoise(dev, h, w, pad):
    net, wh, bh = passing_network(dev, 1, h, w)
    gb = lgx.render_gbuffer_cpu(lgx.make_scene(6, 8, 2), w, h, "f32")
    g = dev.GBufferDev.from_host(gb)
    noisy = np.full((h, w + pad, 4), np.nan, np.float32)
    noisy[:, :w] = np.random.default_rng(w).random((h, w, 4), dtype=np.float32)
    src = torch.from_numpy(noisy).cuda()
    dst = torch.full((h, w + pad, 4), -7.0, device="cuda")
    desc = [lgx.Image(C.c_void_p(t.data_ptr()), w, h, w + pad, lgx.RGBA32F, 0) for t in (src, dst)]
    gd = g.desc
    lgx.check(lgx.lib().lgx_unet_denoise(net.h, C.byref(gd), C.byref(desc[0]), C.byref(desc[1]), dev.stream_handle()),
              "lgx_unet_denoise")
    out = dst.cpu().numpy()
    assert (out[:, w:] == -7.0).all()
    x9 = np.concatenate([noisy[:, :w, :3], gb["depth"][..., None], gb["normal"], gb["albedo"][..., :3]], axis=2)
    assert out[:, :w].tobytes() == head(x9, wh, bh).tobytes()
