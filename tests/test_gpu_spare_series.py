"""The series buffer that a server's engine keeps from a large request goes back
when only smaller ones follow."""
import ctypes as C

import pytest

pytestmark = pytest.mark.gpu


def free_bytes(psx):
    psx.synchronize()
    f = C.c_uint64()
    psx.check(psx.lib().psx_mem_info(C.byref(f), None))
    return f.value


def test_large_buffer_given_back(psx):
    import peasoup_amd.workloads as W
    from peasoup_amd.serve import Server
    n, large, small = 1 << 18, 256, 4
    w = W.Workload("spare", large, n, 64e-6, 41, 5.0, -5.0, 5.0)
    series, dms, args = W.generate_device(w), w.dm_list(), w.search_args()
    with Server(8 << 30, batch=8) as srv:
        def serve(ndm):
            i = srv.submit(args, series, dms[:ndm], accs=[0.0], nsamps=n)
            assert srv.wait(i)["state"] == "done"
            return free_bytes(psx)

        after_large = serve(large)
        assert serve(large) >= after_large - (8 << 20)  # reused
        back = 4 * n * (large - small) - (8 << 20)  # the allocator's granules aside
        assert [serve(small) - after_large >= back for _ in range(10)] == 7 * [False] + 3 * [True]
        again = serve(large)  # kept once more, and taken in time
        for _ in range(7):
            serve(small)
        assert serve(large) >= again - (8 << 20)
        for _ in range(7):
            assert serve(small) - again < back
