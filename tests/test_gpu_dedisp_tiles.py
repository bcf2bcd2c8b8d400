"""Dedispersion at the edges of its kernels' tiles, against the oracle.

The sums are integers and the scaling one float division, so the results
equal the oracle's bit for bit.  Covered: every byte-tile width of the
unpacking pass (16, 32, 64, 128 bytes per sample), samples that end inside
16-sample lanes and 1,024-sample tiles, channel counts off the four-channel
steps, masks, rows staged in LDS by four and by eight waves or read directly by
one and four DM trials per wave, DM counts off those groups, and sums that
leave 16 bits.
"""
import numpy as np
import pytest

from test_gpu_dedisp import _pack

pytestmark = pytest.mark.gpu
f32 = np.float32

CASES = [
    # nbits, nchans, nsamps, ndm, masked channels, all samples at the maximum,
    # largest delay of the list
    (8, 5, 1040, 1, 0, False, 15),           # 16-byte tile, one DM: straight from the rows
    (8, 16, 1 << 14, 3, 16, False, 700),     # every channel masked: zeros
    (2, 64, 187520, 59, 3, False, 1711),     # 16-byte tile, the tutorial's shape
    (1, 256, 4111, 5, 9, False, 37),         # 32-byte tile, 8 channels per byte
    (4, 104, 9001, 6, 1, False, 900),        # 64-byte tile, odd tail
    (8, 130, 5000, 3, 0, False, 1018),       # 128-byte tile with a second, narrow one; the widest spread staged
    (8, 130, 5000, 3, 0, False, 1711),       # beyond it: straight from the rows
    (8, 258, 3000, 5, 0, True, 37),          # 258 x 255 leaves 16 bits
    (4, 4376, 1100, 2, 2, True, 37),         # 4,374 x 15 leaves 16 bits, straight from the rows
    (4, 4376, 1100, 3, 2, True, 37),         # and staged
    (8, 9, 300001, 61, 2, False, 1711),      # eight waves per staged stretch, last group short
    (8, 262, 120007, 70, 1, True, 1711),     # four waves, 32-bit sums, last wave of two DMs
    (8, 259, 300001, 40, 0, True, 1711),     # eight waves, 32-bit sums
    (2, 12, 300001, 41, 1, False, 40000),    # straight from the rows, four DM trials per wave
    (8, 259, 300001, 40, 0, True, 40000),    # the same with 32-bit sums
]


@pytest.mark.parametrize("nbits,nchans,nsamps,ndm,masked,top,reach", CASES)
def test_dedisperse_tiles(psx, orc, nbits, nchans, nsamps, ndm, masked, top, reach):
    import peasoup_amd.sigproc  # noqa: F401  (registers the entry points)
    rng = np.random.default_rng(nbits * 1000 + nchans)
    if top:
        v = np.full((nsamps, nchans), (1 << nbits) - 1)
        v[rng.integers(0, nsamps, 50), rng.integers(0, nchans, 50)] = 0
    else:
        v = rng.integers(0, 1 << nbits, size=(nsamps, nchans))
    packed = _pack(v, nbits)
    dt, f0, df = f32(0.000256), f32(1500.0), f32(-300.0 / nchans)
    table = orc.delay_table(nchans, dt, f0, df)
    dms = np.linspace(0, reach / table[-1], ndm).astype(np.float32)
    km = None
    if masked:
        km = np.ones(nchans, np.int32)
        km[rng.choice(nchans, masked, replace=False)] = 0
    ref = orc.dedisperse(packed, nsamps, nchans, nbits, dms, dt, f0, df, killmask=km)
    nout = ref.shape[1]
    d_in = psx.DeviceArray.from_numpy(packed)
    d_out = psx.DeviceArray.from_numpy(np.full((ndm, nout + 5), -1.0, np.float32))
    work = psx.DeviceArray(int(psx.lib().psx_dedisp_work_bytes(nsamps, nchans, ndm)), np.uint8)
    psx.check(psx.lib().psx_dedisperse(d_in.ptr, nsamps, nchans, nbits, dms.ctypes.data, ndm,
                                       None if km is None else km.ctypes.data, dt, f0, df, d_out.ptr, nout + 5,
                                       work.ptr, None))
    got = d_out.numpy()
    assert np.array_equal(got[:, :nout], ref)
    assert np.all(got[:, nout:] == -1.0)  # nothing past the output samples


@pytest.mark.parametrize("nbits,nchans,nsamps,ndm,masked,top,reach", [
    # runs of 16, 84 and 252 channels whose packed bytes are full, and the
    # 64-channel spans of the staged form's tables: one less, exact, one more
    (4, 34, 3000, 5, 1, True, 300), (4, 64, 3000, 5, 0, True, 300), (4, 66, 3000, 2, 1, True, 300),
    (2, 88, 3000, 5, 4, True, 300), (2, 172, 3000, 7, 3, True, 300), (2, 132, 3000, 2, 3, True, 300),
    (1, 256, 3000, 5, 4, True, 300), (1, 512, 3000, 7, 7, True, 300), (1, 264, 3000, 2, 11, True, 300),
    (8, 63, 3000, 5, 0, True, 300), (8, 128, 3000, 19, 0, True, 300), (8, 129, 3000, 5, 0, True, 300),
    (8, 64, 300001, 40, 1, False, 2000),     # a stretch too long for eight waves: four
])
def test_dedisperse_runs_and_spans(psx, orc, nbits, nchans, nsamps, ndm, masked, top, reach):
    test_dedisperse_tiles(psx, orc, nbits, nchans, nsamps, ndm, masked, top, reach)
