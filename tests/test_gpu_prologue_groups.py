"""The batched search's grouped DM prologues against the Worker's, whose
per-stage kernels the oracle pins: the candidates of every DM are equal, bit
for bit.  Covered: more DMs than a group holds and a short last group, series
on the host and on the device, odd sample counts (unaligned series), series
longer than the FFT, zero padding, a zap list over the spectrum's ends, two
baseline iterations, the shortest length with all three medians, radix-3
lengths, and lengths whose group is one DM.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

ZAPS = [(0.0, 3.0), (50.0, 0.5), (1000.0, 20.0), (7812.0, 5.0)]
CASES = [
    # n, samples, DMs, zap list, on the device, offset
    (256, 256, 3, False, True, 0.0),
    (384, 301, 5, True, False, 0.0),
    (1 << 13, 8191, 67, True, True, 3.0),
    (3 << 12, 3 << 12, 65, False, False, 2.0),
    (1 << 15, 40001, 66, True, True, 1.0),
    (1 << 16, 40001, 5, False, False, 5.0),
    (1 << 24, (1 << 24) - 5, 3, True, True, 0.0),
]


@pytest.mark.parametrize("n,nreal,ndm,zap,device,offset", CASES)
def test_prologue_groups_match_worker(psx, n, nreal, ndm, zap, device, offset):
    import peasoup_amd.workloads as W
    w = W.Workload("g", ndm, n, 64e-6, 1000 + n, 2.0 if n > 4096 else 0.0, -10.0, 10.0, nsamps=nreal)
    if n > 4096:
        w.injections = [W.Injection(int(d), 0.0041 + 0.0003 * d, 5.0, 30.0, 0.1) for d in range(0, ndm, 7)]
    dev = W.generate_device(w) if device and not offset else None
    series = W.generate_host(w) + np.float32(offset)
    if device and dev is None:
        dev = psx.DeviceArray.from_numpy(series)
    args = W.make_search_args(n, 64e-6, acc_start=-10.0, acc_end=10.0, min_snr=5.0 if n > 4096 else 0.5,
                              birdies=ZAPS if zap else None)
    accs = np.array([-10.0, 0.0, 10.0], np.float32)
    ref, _ = W.worker_search(args, series, w.dm_list(), accs, forest=True)
    got, _ = W.batch_search(args, dev if device else series, w.dm_list(), accs, W.make_batch_opts(16), nsamps=nreal,
                            forest=True)
    assert len(ref) > 0
    assert len(got) == len(ref) and np.array_equal(got, ref)
