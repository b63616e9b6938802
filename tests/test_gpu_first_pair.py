"""The first two convolutions' kernel (conv_first_pair_kernel): strips of 30
columns, row pairs, segments of rows per wave.

Against the oracle at extents around a strip (with the network tests'
tolerance, 3e-2 of the correction), and against itself on a shifted crop of
the same records: a pixel further than the network reaches (24) from either
border has the same inputs in another strip, segment and row of a segment, so
its output is the same bit for bit."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

from oracle import unet_ref as U  # noqa: E402

pytestmark = pytest.mark.gpu
REACH = 32


@pytest.fixture(scope="module")
def dev():
    from legitengine_amd import device
    device.require_device()
    return device


def records(seed, n, h, w):
    x = np.zeros((n, h, w, 12), np.float32)
    x[..., :9] = np.random.default_rng(seed).random((n, h, w, 9))
    return x


@pytest.mark.parametrize("n,h,w", [(1, 4, 4), (1, 4, 28), (2, 8, 32), (1, 12, 60), (3, 4, 64), (1, 36, 92)])
def test_against_oracle(dev, n, h, w):
    rng = np.random.default_rng(7)
    layers = [(rng.normal(size=(co, ci, 3, 3)) * np.sqrt(2.0 / (9 * ci)), rng.normal(size=co) * 0.05)
              for ci, co in U.LAYERS]
    flat = U.pack(layers, rng.normal(size=(3, 32)) * 0.3, rng.normal(size=3) * 0.05).astype(np.float32)
    x = records(n * h + w, n, h, w)
    net = dev.UNet(n, h, w)
    net.set(0, flat)
    out = net.forward(torch.from_numpy(x).cuda()).cpu().numpy()
    ref = U.forward(flat.astype(np.float64), x)
    d = (out[..., :3] - x[..., :3]).astype(np.float64) - (ref - x[..., :3])
    assert np.linalg.norm(d) <= 3e-2 * np.linalg.norm(ref - x[..., :3])


@pytest.mark.parametrize("n,h,w,dy,dx", [(1, 128, 160, 4, 4), (2, 108, 240, 8, 28), (1, 1028, 1540, 12, 60)])
def test_shifted_crop(dev, n, h, w, dy, dx):
    x = torch.from_numpy(records(11, n, h, w)).cuda()
    net = dev.UNet(n, h, w, seed=5)
    a = net.forward(x)[:, dy + REACH:h - REACH, dx + REACH:w - REACH]
    b = net.forward(x[:, dy:, dx:].contiguous())[:, REACH:h - dy - REACH, REACH:w - dx - REACH]
    assert a.numel() > 0 and torch.isfinite(a).all()
    assert torch.equal(a, b)
