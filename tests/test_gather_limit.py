"""The gather's march ends at an offset limit instead of the shader's step count
and screen test (indirectLighting.frag:212-228).  The limit restated here in
float64 against that rule, per pixel and direction: a step that only one of
them admits has no side fade, up to the border the FP32 march leaves out
(2^-20 of the extent, where a ramp is below 10 * 2^-20)."""
import numpy as np
import pytest

PI = float(np.float32(3.1415))


@pytest.mark.parametrize("w,h", [(5, 3), (97, 61), (256, 144), (1000, 562), (1279, 719), (2560, 1440)])
@pytest.mark.parametrize("footprint", [1, 4, 32, 256])
@pytest.mark.parametrize("cap", [0, 7])
def test_limit_matches_step_rule(w, h, footprint, cap):
    rng = np.random.default_rng(w * 1000 + footprint)
    n = 4000
    x = rng.integers(0, w, n)
    y = rng.integers(0, h, n)
    edge = rng.integers(0, 4, n)  # half of the pixels next to a border, where the path is shorter than a step
    x = np.where(edge == 0, w - 1 - rng.integers(0, min(w, 4), n), x)
    y = np.where(edge == 1, h - 1 - rng.integers(0, min(h, 4), n), y)
    cx, cy = x + 0.5, y + 0.5
    ang, lin = rng.uniform(0, 2 * PI, n), rng.integers(0, 16, n) / 16.0
    dx, dy = np.cos(ang), np.sin(ang)
    near, ratio = w / 1000.0, 2 * PI / footprint + 1
    path = np.abs(np.minimum(np.maximum(-cx / dx, (w - cx) / dx), np.maximum(-cy / dy, (h - cy) / dy)))
    steps = int(np.log(np.hypot(w, h) / near) / np.log(ratio)) + 2
    steps = max(1, min(steps, cap) if cap else steps)
    off = [near * ratio ** (j + lin) + 1 - near for j in range(steps)] + [np.full(n, np.inf)]
    iters = np.trunc(np.log(path / near) / np.log(ratio)) + 1
    lim = np.where(path >= near, path * ratio ** lin + 1 - near, np.where(path > near / ratio, off[1], 0.0))
    lim = np.minimum(lim, path)
    far = 1 - 2.0 ** -20
    lim32 = np.minimum(lim, np.where(dx > 0, (w * far - cx) / dx, np.inf))
    lim32 = np.minimum(lim32, np.where(dy > 0, (h * far - cy) / dy, np.inf))
    clip = lambda v: np.clip(v * 10, 0, 1)  # noqa: E731
    admitted = 0
    for j in range(steps):
        sx, sy = (cx + dx * off[j]) / w, (cy + dy * off[j]) / h
        rule = (j < iters) & (sx > 0) & (sx < 1) & (sy > 0) & (sy < 1)
        fade = clip(1 - sx) * clip(sx) * clip(1 - sy) * clip(sy)
        assert (fade[rule != (off[j] < lim)] < 1e-12).all()
        assert (fade[rule != (off[j] < lim32)] <= 10 * 2.0 ** -20).all()
        admitted += int(rule.sum())
    assert admitted > 0
