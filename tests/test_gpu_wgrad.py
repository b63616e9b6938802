"""The weight gradient's division of the pixels: 32-column strips, rows in even
shares over the waves, shares that end inside a strip, an image or a row list
shorter than the waves.

Against the oracle with the network tests' tolerances (5e-2 of the whole
gradient, 0.15 of a layer's: activations and their gradients are BF16), and
against itself: n copies of one image (n a power of two) have the same BF16
activations and gradients of activations that are the single image's divided
by n, exactly, so the sums differ only by their FP32 order: 1e-5 of a layer's
norm (2^-24 times the square root of the 10^4 to 10^6 terms a weight sums)."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

from oracle import unet_ref as U  # noqa: E402

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def dev():
    from legitengine_amd import device
    device.require_device()
    return device


def case(seed, n, h, w):
    rng = np.random.default_rng(seed)
    layers = [(rng.normal(size=(co, ci, 3, 3)) * np.sqrt(2.0 / (9 * ci)), rng.normal(size=co) * 0.05)
              for ci, co in U.LAYERS]
    flat = U.pack(layers, rng.normal(size=(3, 32)) * 0.3, rng.normal(size=3) * 0.05).astype(np.float32)
    x = np.zeros((n, h, w, 12), np.float32)
    x[..., :9] = rng.random((n, h, w, 9))
    t = np.zeros((n, h, w, 4), np.float32)
    t[..., :3] = rng.random((n, h, w, 3)) * 2.0
    return flat, x, t


def gradient(dev, flat, x, t):
    net = dev.UNet(*x.shape[:3])
    net.set(0, flat)
    net.backward(torch.from_numpy(x).cuda(), torch.from_numpy(t).cuda())
    return net.get(1)[0].astype(np.float64)


def rel(a, b):
    return np.linalg.norm(a - b) / np.linalg.norm(b)


def layers_of(g):
    off = 0
    for ci, co in U.LAYERS:
        yield g[off:off + co * ci * 9]
        yield g[off + co * ci * 9:off + co * ci * 9 + co]
        off += co * ci * 9 + co


@pytest.mark.parametrize("n,h,w", [(1, 8, 36), (3, 12, 32), (1, 68, 4), (2, 36, 68)])
def test_against_oracle(dev, n, h, w):
    flat, x, t = case(n + h + w, n, h, w)
    g = gradient(dev, flat, x, t)
    ref = U.backward(flat.astype(np.float64), x, t, "l1")[1]
    assert rel(g, ref) <= 5e-2
    for a, b in zip(layers_of(g), layers_of(ref)):
        assert rel(a, b) <= 0.15


@pytest.mark.parametrize("n,h,w", [(2, 4, 4), (4, 20, 100), (16, 64, 64), (2, 260, 516), (8, 132, 36)])
def test_copies_of_one_image(dev, n, h, w):
    flat, x, t = case(5, 1, h, w)
    one = gradient(dev, flat, x, t)
    many = gradient(dev, flat, np.repeat(x, n, 0), np.repeat(t, n, 0))
    for a, b in zip(layers_of(many), layers_of(one)):
        assert rel(a, b) <= 1e-5
