"""psx_remove_baseline's loop on series whose every step counts, against the
oracle: one to five steps and the cap of 102, where a step less shows.

Two kinds of samples: a few so large that a mean is lost in their rounding, in
pairs of opposite sign, and small ones that take every mean.  With one in 16
large, a step leaves a 16th of the mean behind, until it is at most 5e-7 n.
"""
import numpy as np
import pytest

f32 = np.float32
N = 100003  # the loop stops at a mean of 0.05


def series(steps):
    if steps == 102:  # all but five are large: the mean stays near 75
        x = (2.0 ** 32 * (1 - np.arange(N) % 2 * 2)).astype(f32)
        x[-5:] = 75 * N / 5
        return x
    x = np.full(N, 0.7 * 16.0 ** (steps - 2) * 16 / 15, f32)
    x += f32(0.25) * (np.arange(N) % 3 - 1).astype(f32)
    big = np.random.default_rng(steps).permutation(N)[:N // 32 * 2]
    x[big[::2]] = 2.0 ** (21 + 4 * (steps - 1))
    x[big[1::2]] = -x[big[::2]]
    return x


def loop(x, most=1000):
    """The loop and the tolerance on its result: a mean is off by its rounding
    and by that of up to 32 additions of doubles in a row, on either side, and a
    sample by its own rounding, in each step."""
    y, steps = x.copy(), 0
    tol = np.zeros(x.size)
    while True:
        mean = f32(f32(y.sum(dtype=np.float64)) / f32(y.size))
        off = np.spacing(abs(mean)) + 2 * 32 * 2.0 ** -53 * np.abs(y).sum(dtype=np.float64) / y.size
        y = (y - mean).astype(f32)
        tol += off + np.spacing(np.abs(y))
        steps += 1
        if steps >= most or steps > 101 or not abs(float(mean)) > 5e-7 * y.size:
            return y, steps, tol


@pytest.mark.parametrize("steps", [1, 2, 3, 4, 5, 102])
def test_every_step_counts(orc, steps):
    x = series(steps)
    ref = orc.remove_baseline(x.copy())
    y, n, tol = loop(x)
    assert n == steps and np.all(np.abs(y - ref) <= tol)
    if steps > 1:
        early, _, _ = loop(x, steps - 1)
        assert np.max(np.abs(early - ref) / tol) > 3


@pytest.mark.gpu
@pytest.mark.parametrize("steps", [1, 2, 3, 4, 5, 102])
def test_remove_baseline_steps(psx, orc, steps):
    x = series(steps)
    _, _, tol = loop(x)
    d_x = psx.DeviceArray.from_numpy(x)
    d_w = psx.DeviceArray(int(psx.lib().psx_reduce_work_bytes()), np.uint8)
    psx.check(psx.lib().psx_remove_baseline(d_x.ptr, N, d_w.ptr, None))
    assert np.all(np.abs(d_x.numpy() - orc.remove_baseline(x.copy())) <= tol)
