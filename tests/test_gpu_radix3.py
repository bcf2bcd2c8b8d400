"""Transforms of 3*2^k points in every tile: radices 24, 12 or 6 first, then
8s; 24 points per thread.  Plain plans against the double DFT, contiguous-row
kernels (one or several tiles per workgroup) against the natural layout."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

COLUMNS = [(48, 16), (96, 16), (192, 16), (384, 16), (768, 16), (96, 8), (192, 8), (384, 8), (768, 8), (1536, 8),
           (384, 4), (768, 4), (1536, 4), (3072, 4)]
SINGLE = [(12, 1), (24, 1), (48, 1), (96, 1), (192, 1), (384, 1), (768, 1), (1536, 1), (3072, 1)]


@pytest.mark.parametrize("decomp", [[s] for s in SINGLE] + [[c, (64, 16)] for c in COLUMNS] +
                         [[(64, 16), c] for c in COLUMNS])
def test_radix3_passes_vs_exact(psx, decomp):
    n, batch = 2 * int(np.prod([L for L, _ in decomp])), 3
    x = np.random.default_rng(n).standard_normal((batch, n)).astype(np.float32)
    plan = psx.FFTPlan(n, psx.PSX_FFT_R2C, batch=batch, decomp=decomp)
    d_x = psx.DeviceArray.from_numpy(x)
    d_X = psx.DeviceArray(batch * (n // 2 + 1), np.complex64)
    plan.execute(d_x, d_X)
    ref = np.fft.rfft(x.astype(np.float64))
    # max over rms, as for every other decomposition
    assert np.max(np.abs(d_X.numpy().reshape(ref.shape) - ref)) < 2e-6 * np.sqrt(np.mean(np.abs(ref) ** 2))


@pytest.mark.parametrize("n,decomp", [(3 << 15, [(64, 16), (768, 8)]), (3 << 18, [(256, 16), (1536, 4)]),
                                      (3 << 18, [(256, 16), (1536, 8)]), (3 << 20, [(512, 16), (3072, 4)])])
@pytest.mark.parametrize("batch", [2, 24])
def test_radix3_rows_equal_natural(psx, n, decomp, batch):
    import peasoup_amd.workloads as W
    w = W.Workload("rows", 1, n, 64e-6, 77, 0.0, -50.0, 50.0, injections=[W.Injection(0, 0.0123, 20.0, 15.0, 0.2)])
    series = W.generate_host(w)
    accs = np.linspace(-50, 50, 29).astype(np.float32)  # a partial batch at the end
    got = [W.batch_search(w.search_args(), series, w.dm_list(), accs,
                          W.make_batch_opts(batch, decomp=decomp, spectrum_layout=lay), forest=True)[0]
           for lay in (W.SPECTRUM_NATURAL, W.SPECTRUM_ROWS)]
    assert len(got[0]) > 0
    key = lambda c: tuple(c[k].item() for k in ("dm_idx", "acc", "nh", "freq", "snr", "nassoc"))
    assert sorted(map(key, got[0])) == sorted(map(key, got[1]))
