"""Series buffers that outlive a call: those of the batched search (with its
kept engine) and those of the server's finished requests."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def key(cands):
    return sorted(tuple(c[k].item() for k in ("dm_idx", "acc", "nh", "freq", "snr", "nassoc")) for c in cands)


def workload(W, n, ndm, seed):
    return W.Workload("kept", ndm, n, 64e-6, seed, 5.0, -50.0, 50.0,
                      injections=[W.Injection(ndm - 1, 0.0123 + 1e-4 * seed, 20.0, 40.0, 0.2)])


def test_batch_search_keeps_and_regrows(psx):
    import peasoup_amd.workloads as W
    n = 1 << 15
    kept, fresh = W.make_batch_opts(8, keep_engine=True), W.make_batch_opts(8)
    args = W.make_search_args(n, 64e-6, acc_start=-50.0, acc_end=50.0)
    # more DMs, fewer, an engine of its own between, nothing kept, a short series
    for seed, ndm, nreal, release in [(1, 2, n, False), (2, 70, n, False), (3, 1, n, False), (4, 3, n, True),
                                      (5, 70, n - 4097, False), (6, 2, n - 1, False)]:
        w = workload(W, n, ndm, seed)
        series = np.ascontiguousarray(W.generate_host(w)[:, :nreal])
        if release:
            psx.check(psx.lib().psx_batch_release())
        got, _ = W.batch_search(args, series, w.dm_list(), None, kept, forest=True)
        ref, _ = W.batch_search(args, series, w.dm_list(), None, fresh, forest=True)
        assert len(ref) > 0 and key(got) == key(ref), seed
    psx.check(psx.lib().psx_batch_release())


@pytest.mark.parametrize("mixed", [False, True])
def test_server_reuses_series_buffers(psx, mixed):
    import peasoup_amd.workloads as W
    from peasoup_amd.serve import DISPATCH_MIXED_GRAPH, DISPATCH_STREAMS, Server
    shapes = [(1 << 15, 3, 11), (1 << 15, 3, 12), (1 << 15, 5, 13), (1 << 16, 2, 14), (1 << 15, 3, 15), (1 << 16, 2, 16)]
    ws = [workload(W, *s) for s in shapes]
    series = [W.generate_host(w) for w in ws]
    alone = [W.batch_search(w.search_args(), x, w.dm_list(), None, W.make_batch_opts(8))[0] for w, x in zip(ws, series)]
    with Server(8 << 30, batch=8, dispatch=DISPATCH_MIXED_GRAPH if mixed else DISPATCH_STREAMS) as srv:
        for rounds in range(2):  # one after the other, then all at once
            ids = []
            for w, x in zip(ws, series):
                ids.append(srv.submit(w.search_args(), x, w.dm_list()))
                if rounds == 0:
                    assert srv.wait(ids[-1])["state"] == "done"
            for i, ref in zip(ids, alone):
                assert srv.wait(i)["state"] == "done"
                assert len(ref) > 0 and key(srv.result(i)) == key(ref)
        assert srv.stats()["failed"] == 0


def test_spare_buffers_yield_to_the_budget(psx):
    """A budget for one engine and one request's series: the spare buffer of
    the first never keeps the next from being admitted."""
    import peasoup_amd.workloads as W
    from peasoup_amd.serve import Server
    small, large = workload(W, 1 << 15, 2, 21), workload(W, 1 << 15, 64, 22)
    x = {w.ndm: W.generate_host(w) for w in (small, large)}
    for nbytes in range(64 << 20, 1 << 30, 1 << 20):  # the least budget that takes the larger request
        with Server(nbytes, batch=8) as srv:
            try:
                i = srv.submit(large.search_args(), x[64], large.dm_list())
            except psx.PsxError:
                continue
            assert srv.wait(i)["state"] == "done"
            for w in (small, large, small, large):
                i = srv.submit(w.search_args(), x[w.ndm], w.dm_list())
                assert srv.wait(i)["state"] == "done"
                assert srv.stats()["used_bytes"] <= nbytes
            return
    assert False, "no budget taken"
