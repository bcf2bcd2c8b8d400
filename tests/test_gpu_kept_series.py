"""The series that a batched search with keep_engine leaves in device memory are
given back when an allocation of the library finds none."""
import ctypes as C

import pytest

pytestmark = pytest.mark.gpu


def free_bytes(psx):
    psx.synchronize()
    f, t = C.c_uint64(), C.c_uint64()
    psx.check(psx.lib().psx_mem_info(C.byref(f), C.byref(t)))
    return f.value, t.value


def test_kept_series_yield_to_allocations(psx):
    import peasoup_amd.workloads as W
    n, ndm = 1 << 20, 32
    w = W.Workload("kept", ndm, n, 64e-6, 31, 5.0, -5.0, 5.0,
                   injections=[W.Injection(ndm - 1, 0.0123, 0.0, 40.0, 0.2)])
    series, args = W.generate_device(w), w.search_args()
    kept = W.make_batch_opts(32, keep_engine=True)
    run = lambda: W.batch_search(args, series, w.dm_list(), [0.0], kept, nsamps=n)[0]
    psx.check(psx.lib().psx_batch_release())
    first = run()
    before, total = free_bytes(psx)
    p = C.c_void_p()
    assert psx.lib().psx_malloc(C.byref(p), 2 * total) != 0 and not p.value  # more than the device has
    after, _ = free_bytes(psx)
    assert after - before >= 4 * n * ndm - (8 << 20)  # the series are gone, the allocator's granules aside
    again = run()  # with the same engine
    assert len(first) > 0 and (first == again).all()
    psx.check(psx.lib().psx_batch_release())
