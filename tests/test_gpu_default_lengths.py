"""Default two-pass plans follow one rule over the lengths: before the rows, the
largest power of two that is at most 1,024 and no longer than they are, with 512
for 256 before longer rows; no length has a plan of its own."""
import re

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def split(M):
    m2 = 1024
    while M % m2 or M // m2 < m2:
        m2 //= 2
    m1 = M // m2
    return (512, m1 // 2) if m2 == 256 and m1 > 256 else (m2, m1)


@pytest.mark.parametrize("n", [1 << k for k in range(14, 24)] + [3 << k for k in range(14, 22)])
def test_split_follows_the_rule(psx, n):
    plan = psx.FFTPlan(n).describe()
    got = tuple(int(x) for x in re.search(r"passes=(\d+)/C\d+x(\d+)/C\d+ ", plan).groups())
    assert got == split(n // 2), plan


@pytest.mark.parametrize("batch", [1, 5])
def test_rows_of_3072_vs_exact(psx, batch):
    n = 3 << 21
    x = np.random.default_rng(n + batch).standard_normal((batch, n)).astype(np.float32)
    r2c, c2r = psx.FFTPlan(n, psx.PSX_FFT_R2C, batch=batch), psx.FFTPlan(n, psx.PSX_FFT_C2R, batch=batch)
    d_x, d_X = psx.DeviceArray.from_numpy(x), psx.DeviceArray(batch * (n // 2 + 1), np.complex64)
    d_y = psx.DeviceArray(batch * n, np.float32)
    r2c.execute(d_x, d_X)
    ref = np.fft.rfft(x.astype(np.float64))
    # max over rms, as for every other plan
    assert np.max(np.abs(d_X.numpy().reshape(ref.shape) - ref)) < 2e-6 * np.sqrt(np.mean(np.abs(ref) ** 2))
    c2r.execute(d_X, d_y)
    assert np.max(np.abs(d_y.numpy().reshape(x.shape) / n - x)) < 4e-6  # there and back
