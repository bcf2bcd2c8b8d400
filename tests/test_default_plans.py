"""Default FFT plans around the lengths whose strided pass of 256 points gives
way to one of 512 before shorter rows."""
import numpy as np
import pytest

import peasoup_amd as P

SIZES = [(1 << 17, "256/C8x256"), (1 << 18, "512/C8x256"), (3 << 16, "512/C8x192"), (3 << 17, "512/C8x384"),
         (1 << 19, "512/C8x512")]


@pytest.mark.parametrize("n", [n for n, _ in SIZES])
@pytest.mark.parametrize("batch", [1, 3, 8, 64])
def test_layouts_in_bounds(n, batch):
    for kind in (P.PSX_FFT_R2C, P.PSX_FFT_C2R):
        assert P.lib().psx_fft_layout_check(n, kind, batch, 0, None, None) == 0, P.lib().psx_last_error_string()


@pytest.mark.gpu
@pytest.mark.parametrize("n,plan", SIZES)
@pytest.mark.parametrize("batch", [1, 5])
def test_default_plans_vs_exact(psx, n, plan, batch):
    x = np.random.default_rng(n + batch).standard_normal((batch, n)).astype(np.float32)
    r2c, c2r = psx.FFTPlan(n, psx.PSX_FFT_R2C, batch=batch), psx.FFTPlan(n, psx.PSX_FFT_C2R, batch=batch)
    if batch == 1:
        assert plan in r2c.describe(), r2c.describe()
    d_x, d_X = psx.DeviceArray.from_numpy(x), psx.DeviceArray(batch * (n // 2 + 1), np.complex64)
    d_y = psx.DeviceArray(batch * n, np.float32)
    r2c.execute(d_x, d_X)
    ref = np.fft.rfft(x.astype(np.float64))
    # max over rms, as for every other plan
    assert np.max(np.abs(d_X.numpy().reshape(ref.shape) - ref)) < 2e-6 * np.sqrt(np.mean(np.abs(ref) ** 2))
    c2r.execute(d_X, d_y)
    assert np.max(np.abs(d_y.numpy().reshape(x.shape) / n - x)) < 4e-6  # there and back
