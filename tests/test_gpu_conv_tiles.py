"""The convolution tiles with direct loads to LDS (conv3x3_dma_kernel) against
tile 0 (registers only): every output is accumulated in the same order, so
forward, gradients and denoised images are equal bit for bit.

Extents around the tiles' 8 or 16 rows x 32 pixels and their halves and
quarters (the layers' resolutions): smaller than one tile, exact, one step
over, several images, and one where every workgroup walks several tiles at
all three resolutions."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

from legitengine_amd import lgx  # noqa: E402
from oracle import unet_ref as U  # noqa: E402

pytestmark = pytest.mark.gpu

COUTS = [co for _, co in U.LAYERS]
CINS = [32, 32, 32, 64, 64, 128, 192, 64, 96, 32]  # padded input channels
FIRST = {32: 10, 64: 11, 96: 5, 128: 6, 192: 4}  # the first direct-load tile of a channel count


@pytest.fixture(scope="module")
def dev():
    from legitengine_amd import device
    device.require_device()
    return device


def picks(channels, k):
    counts = [lgx.lib().lgx_unet_conv_tiles(c) for c in channels]
    return [min(FIRST[c] + k, n - 1) for c, n in zip(channels, counts)]


def inputs(n, h, w):
    rng = np.random.default_rng(n * h + w)
    x = torch.from_numpy(rng.standard_normal((n, h, w, 12)).astype(np.float32)).cuda()
    t = torch.from_numpy(rng.random((n, h, w, 4)).astype(np.float32)).cuda()
    return x, t


@pytest.mark.parametrize("n,h,w", [(1, 4, 4), (2, 8, 32), (1, 12, 36), (1, 36, 68), (3, 16, 128), (2, 60, 132)])
def test_forward_and_gradients_equal_register_tiles(dev, n, h, w):
    x, t = inputs(n, h, w)
    net = dev.UNet(n, h, w, seed=3)
    net.set_tiles([0] * 10, [0] * 10)
    out = net.forward(x).cpu().numpy()
    net.backward(x, t)
    convs = sum(co * ci * 9 + co for ci, co in U.LAYERS)  # (the head's gradients are FP32 atomic sums)
    grad = net.get(1)[0][:convs]
    assert np.isfinite(out).all() and np.abs(grad).max() > 0
    for k in range(2):
        net.set_tiles(picks(COUTS, k), picks(CINS, k))
        assert net.forward(x).cpu().numpy().tobytes() == out.tobytes(), k
        net.backward(x, t)
        assert net.get(1)[0][:convs].tobytes() == grad.tobytes(), k


@pytest.mark.parametrize("h,w", [(4, 8), (44, 100), (1028, 1540)])
def test_denoise_equals_register_tiles(dev, h, w):
    gb = lgx.render_gbuffer_cpu(lgx.make_scene(6, 8, 2), w, h, "mixed")
    g = dev.GBufferDev.from_host(gb)
    noisy = dev.DImage.from_numpy(np.random.default_rng(2).random((h, w, 4)).astype(np.float32), lgx.RGBA32F)
    net = dev.UNet(1, h, w, seed=4)
    net.set_tiles([0] * 10, [0] * 10)
    ref = net.denoise(g, noisy).numpy()
    for k in range(2):
        net.set_tiles(picks(COUTS, k), [0] * 10)
        assert net.denoise(g, noisy).numpy().tobytes() == ref.tobytes(), k


@pytest.mark.parametrize("n,h,w", [(1, 4, 4), (1, 400, 400), (1, 448, 896), (1, 800, 1024)])
def test_default_tiles(dev, n, h, w):
    """A new network's tiles, below and above the rule's pixel counts (40000
    and 200000 at a layer's resolution), are offered ones and change no bit."""
    x, _ = inputs(n, h, w)
    net = dev.UNet(n, h, w, seed=3)
    f, d = net.tiles()
    for t, c in zip(f + d, COUTS + CINS):
        assert 0 <= t < lgx.lib().lgx_unet_conv_tiles(c)
    out = net.forward(x).cpu().numpy()
    net.set_tiles([0] * 10, [0] * 10)
    assert net.forward(x).cpu().numpy().tobytes() == out.tobytes()
