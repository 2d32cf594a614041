"""The bound by which perturbation blocks leave their rebase tests out: with |d| + |dc| just
below its reciprocal, in any direction and split, no test of the block's 32 steps may fire,
in either precision (numpy restatement of quiet_bound and of the kernel's step)."""
import numpy as np
import pytest

import _oracle

STEPS = 32


def quiet_bounds(z, starts):
    """quiet_bound of the blocks from `starts`, in FP32 as the kernel computes it."""
    f, u, c = np.float32, np.ones(len(starts), np.float32), np.zeros(len(starts), np.float32)
    with np.errstate(all="ignore"):
        for k in range(STEPS):
            x, y = z[starts + k, 0].astype(f), z[starts + k, 1].astype(f)
            r = np.sqrt(x * x + y * y)
            c = np.where(r > f(1e-6), np.fmax(c, f(4.16) * u / r), f(np.inf))
            u = f(2.35) * r * u + f(1.04)
    return c


@pytest.mark.parametrize("centre", [(-0.743643887037151, 0.131825904205330), (-0.25, 0.125),
                                    (-1.7548776662466927, 0.0), (-0.1225, 0.7448), (0.2501, 0.0),
                                    (0.0, 1.0), (-2.0, 0.0), (0.0, 0.0)])
@pytest.mark.parametrize("precision", [32, 64])
def test_no_test_fires_below_the_bound(centre, precision):
    real = np.float32 if precision == 32 else np.float64
    z, last = _oracle.reference_orbit(*centre, 2000, 256.0, precision)
    starts = np.arange(0, last // STEPS * STEPS, STEPS)
    bounds = quiet_bounds(z, starts)
    starts, bounds = starts[np.isfinite(bounds)], bounds[np.isfinite(bounds)]
    assert len(starts) > 0 or centre in ((0.0, 0.0), (-1.7548776662466927, 0.0))
    rng = np.random.default_rng(7)
    n = 400
    for start, bound in zip(starts, bounds):
        a, b, part = rng.uniform(0, 2 * np.pi, n), rng.uniform(0, 2 * np.pi, n), rng.random(n)
        part[:20], part[20:40] = 0, 1
        d = np.stack([np.cos(a), np.sin(a)]) * part
        dc = np.stack([np.cos(b), np.sin(b)]) * (1 - part)
        scale = 0.9999 / float(bound) / (np.abs(d).sum(0) + np.abs(dc).sum(0))
        (dx, dy), (ex, ey) = (d * scale).astype(real), (dc * scale).astype(real)
        for k in range(STEPS):
            x, y, h = (real(v) for v in z[start + k, :3])
            assert not np.any(x * dx + y * dy < -h)
            assert np.all(np.hypot(dx, dy) <= 0.26 * np.hypot(x, y))
            ax, ay = 2 * x + dx, 2 * y + dy
            dx, dy = ax * dx - ay * dy + ex, ax * dy + ay * dx + ey
