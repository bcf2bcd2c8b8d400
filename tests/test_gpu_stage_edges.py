"""Per-stage kernels at the edges of their tiles, against the oracle.

Peak compaction (4,096-bin tiles of 16-byte loads from any start), harmonic
sums (512 bins per wave, then bin by bin), the running median (2,000 bins per
workgroup, three zones) and the baseline loop (two iterations per look).
"""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu
f32 = np.float32


def dev(psx, a):
    return psx.DeviceArray.from_numpy(np.ascontiguousarray(a))


def find_peaks(psx, p, start, end, thr, cap):
    d_p = dev(psx, p)
    d_i, d_s = dev(psx, np.full(cap + 1, -7, np.int32)), dev(psx, np.full(cap + 1, -7, f32))
    d_c = dev(psx, np.zeros(1, np.uint32))
    work = psx.DeviceArray(int(psx.lib().psx_find_peaks_work_bytes(end - start)), np.uint8)
    psx.check(psx.lib().psx_find_peaks(d_p.ptr, start, end, thr, d_i.ptr, d_s.ptr, cap, d_c.ptr, work.ptr, None))
    return d_i.numpy(), d_s.numpy(), int(d_c.numpy()[0])


@pytest.mark.parametrize("start,end,thr,cap", [
    (0, 1, -9.0, 4), (3, 4099, 0.0, 5000), (1, 4097, 2.0, 500), (2, 4099, -9.0, 4097), (5, 8195, 3.0, 100),
    (7, 100003, 1.0, 20000), (4095, 4097, -9.0, 2), (0, 100003, 9.0, 10), (13, 60001, 0.0, 1000),
])
def test_peak_tiles(psx, start, end, thr, cap):
    p = np.random.default_rng(end).standard_normal(100003).astype(f32)
    p[::997] = np.nan  # never above a threshold
    idx, snr, count = find_peaks(psx, p, start, end, thr, cap)
    want = np.flatnonzero(p[start:end] > f32(thr)) + start
    assert count == want.size
    m = min(cap, want.size)
    assert np.array_equal(idx[:m], want[:m]) and np.array_equal(snr[:m], p[want[:m]])
    assert np.all(idx[m:] == -7) and np.all(snr[m:] == -7)  # nothing past the survivors or the capacity


@pytest.mark.parametrize("nfolds", [1, 2, 3, 4, 5])
@pytest.mark.parametrize("nb", [1, 511, 512, 513, 2048, 2049, 5000])
def test_harmonic_tiles(psx, orc, nfolds, nb):
    P = np.random.default_rng(nb).standard_normal(nb).astype(f32)
    d_P = dev(psx, P)
    folds = [dev(psx, np.full(nb + 1, -7, f32)) for _ in range(nfolds)]
    arr = (C.c_void_p * nfolds)(*[f.ptr for f in folds])
    psx.check(psx.lib().psx_harmonic_sum(d_P.ptr, arr, nfolds, nb, None))
    ref = orc.harmonic_sum(P, nfolds)
    for k in range(nfolds):
        got = folds[k].numpy()
        assert np.array_equal(got[:nb], ref[k]) and got[nb] == -7


@pytest.mark.parametrize("nb", [125, 129, 624, 1999, 2000, 2001, 2005, 4003, 10007])
@pytest.mark.parametrize("bw", [1e-5, 4e-4, 3e-3, 0.2, 9.0])
def test_median_zones(psx, orc, nb, bw):
    A = np.abs(np.random.default_rng(nb).standard_normal(nb)).astype(f32)
    d_A, d_m = dev(psx, A), dev(psx, np.full(nb, -7, f32))
    d_w = psx.DeviceArray(int(psx.lib().psx_deredden_work_floats(nb)))
    psx.check(psx.lib().psx_deredden_median(d_A.ptr, nb, bw, 0.05, 0.5, d_m.ptr, d_w.ptr, None))
    # the oracle's scrunches and stretches, composed by zone (its own
    # calculate_median copies like the reference, whose second copy needs
    # pos5 + pos25 <= nb)
    m5 = orc.median_scrunch5(A)
    m25 = orc.median_scrunch5(m5)
    m125 = orc.median_scrunch5(m25)
    z1, z2 = (min(int(float(f32(b)) / bw), nb) for b in (0.05, 0.5))
    ref = orc.linear_stretch(m125, nb)
    ref[:z2] = orc.linear_stretch(m25, nb)[:z2]
    ref[:z1] = orc.linear_stretch(m5, nb)[:z1]
    assert np.array_equal(d_m.numpy(), ref)


@pytest.mark.parametrize("n,offset", [(1000, 0.0), (131, 3.0), (100001, 5.0), (1 << 17, 2.0 ** 22)])
def test_baseline_loop(psx, n, offset):
    """The loop restated in numpy (float64 sums, float32 means): both end with
    a mean at most 5e-7 n from zero, taken from the same series."""
    x = (np.random.default_rng(n).standard_normal(n) + offset).astype(f32)
    d_x = dev(psx, x)
    d_w = psx.DeviceArray(int(psx.lib().psx_reduce_work_bytes()), np.uint8)
    psx.check(psx.lib().psx_remove_baseline(d_x.ptr, n, d_w.ptr, None))
    ref, steps = x.copy(), 0
    while True:
        mean = f32(f32(ref.sum(dtype=np.float64)) / f32(n))
        ref = (ref - mean).astype(f32)
        steps += 1
        if steps > 101 or not abs(float(mean)) > 5e-7 * n:
            break
    # the sums' order moves a mean by at most an ulp in each iteration
    assert np.max(np.abs(d_x.numpy() - ref)) <= 4 * np.spacing(f32(max(1.0, offset)))


@pytest.mark.parametrize("n,batch", [(16, 3), (24, 2), (192, 1), (1 << 14, 5), (3 << 13, 3), (3 << 20, 1)])
def test_c2r_pairs(psx, orc, n, batch):
    rng = np.random.default_rng(n)
    X = (rng.standard_normal((batch, n // 2 + 1)) + 1j * rng.standard_normal((batch, n // 2 + 1))).astype(np.complex64)
    X[:, 0] = X[:, 0].real
    X[:, -1] = X[:, -1].real
    plan = psx.FFTPlan(n, psx.PSX_FFT_C2R, batch)
    d_X, d_x = dev(psx, X), psx.DeviceArray((batch, n))
    plan.execute(d_X, d_x)
    ref = np.fft.irfft(X.astype(np.complex128), n, axis=1) * n
    assert np.max(np.abs(d_x.numpy() - ref)) <= 2e-6 * np.sqrt(np.mean(ref ** 2)) * np.log2(n)


@pytest.mark.parametrize("ranges,thr,cap,nhead", [
    ([(0, 4097), (3, 3), (7, 100003), (100002, 100003), (0, 4096)], 2.0, 500, 16),
    ([(0, 100003)] * 8, 0.0, 70000, 300), ([(5, 5), (9, 2)], 0.0, 10, 4), ([(13, 60001)], 3.0, 0, 1000),
    ([(0, 1), (4095, 8193)], -9.0, 5000, 0),
])
def test_peaks_of_several_spectra(psx, ranges, thr, cap, nhead):
    n = len(ranges)
    ps = [np.random.default_rng(y).standard_normal(100003).astype(f32) for y in range(n)]
    d_ps = [dev(psx, p) for p in ps]
    d_i, d_s = dev(psx, np.full(n * cap + 1, -7, np.int32)), dev(psx, np.full(n * cap + 1, -7, f32))
    d_h = dev(psx, np.full(n * (1 + 2 * nhead) + 1, 0xC0E00000, np.uint32))  # -7.0f
    work = psx.DeviceArray(sum(int(psx.lib().psx_find_peaks_work_bytes(max(b - a, 0))) for a, b in ranges), np.uint8)
    a64 = lambda k: (C.c_int64 * n)(*[r[k] for r in ranges])
    psx.check(psx.lib().psx_find_peaks_spectra((C.c_void_p * n)(*[d.ptr for d in d_ps]), a64(0), a64(1), n, thr,
                                               d_i.ptr, d_s.ptr, cap, d_h.ptr, nhead, work.ptr, None))
    idx, snr, head = d_i.numpy(), d_s.numpy(), d_h.numpy()
    assert idx[-1] == -7 and snr[-1] == -7 and head[-1] == 0xC0E00000
    hidx = head[n:n + n * nhead].view(np.int32).reshape(n, nhead)
    hsnr = head[n + n * nhead:-1].view(f32).reshape(n, nhead)
    for y, (a, b) in enumerate(ranges):
        want = np.flatnonzero(ps[y][a:b] > f32(thr)) + a
        assert head[y] == want.size
        m = min(cap, want.size)
        assert np.array_equal(idx[y * cap:y * cap + m], want[:m]) and np.all(idx[y * cap + m:(y + 1) * cap] == -7)
        assert np.array_equal(snr[y * cap:y * cap + m], ps[y][want[:m]])
        m = min(nhead, want.size)
        assert np.array_equal(hidx[y, :m], want[:m]) and np.array_equal(hsnr[y, :m], ps[y][want[:m]])
        assert np.all(hsnr[y, m:] == -7)


def test_peaks_of_several_spectra_refusals(psx):
    d = dev(psx, np.zeros(64, f32))
    ptr, at = (C.c_void_p * 9)(*[d.ptr] * 9), (C.c_int64 * 9)()
    call = lambda n, i, h: psx.lib().psx_find_peaks_spectra(ptr, at, at, n, 0.0, i, i, 1, h, 1, d.ptr, None)
    assert call(0, d.ptr, d.ptr) != 0 and call(9, d.ptr, d.ptr) != 0
    assert call(1, None, d.ptr) != 0 and call(1, d.ptr, None) != 0
