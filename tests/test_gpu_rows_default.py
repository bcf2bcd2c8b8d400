"""The row layout asked for without a decomposition, at lengths whose default
plan has none: the two passes with the longest last one, as if given."""
import pytest

from test_gpu_batch import _plan_desc, same

pytestmark = pytest.mark.gpu


def workload(W, n):
    return W.Workload("rows", 2, n, 64e-6, 0x5EA5D0 + n % 97, 0.0, -50.0, 50.0,
                      injections=[W.Injection(1, 0.0123, 20.0, 25.0, 0.2)])


@pytest.mark.parametrize("n,batch,decomp", [
    (1 << 14, 8, [(32, 16), (256, 16)]), (1 << 15, 24, [(32, 16), (512, 16)]), (3 << 15, 64, [(32, 16), (1536, 8)]),
    (1 << 17, 1, [(32, 16), (2048, 8)]), (3 << 16, 16, [(32, 16), (3072, 4)]), (1 << 18, 2, [(32, 16), (4096, 4)]),
    (3 << 17, 64, [(48, 16), (4096, 4)]), (1 << 19, 1, [(64, 16), (4096, 4)]), (3 << 18, 1, [(96, 16), (4096, 4)]),
])
def test_rows_without_a_decomposition(psx, n, batch, decomp):
    import peasoup_amd.workloads as W
    w = workload(W, n)
    series = W.generate_host(w)
    accs = W.accel_list(w.size, w.tsamp, w.acc_lo, w.acc_hi)
    accs = accs[:: max(1, accs.size // 8)]
    rows = W.make_batch_opts(batch, spectrum_layout=W.SPECTRUM_ROWS)
    nat = W.make_batch_opts(batch, decomp=decomp, spectrum_layout=W.SPECTRUM_NATURAL)
    plan = "x".join("%d/C%d" % p for p in decomp) + " rows"
    assert _plan_desc(psx, W, w, series[0], accs, rows).endswith(plan)
    ref, _ = W.batch_search(w.search_args(), series, w.dm_list(), accs, nat, forest=True)
    got, _ = W.batch_search(w.search_args(), series, w.dm_list(), accs, rows, forest=True)
    assert len(ref) > 0 and same(got, ref)


@pytest.mark.parametrize("n", [1 << 12, 1 << 16])  # one pass; rows of 1,024 points in 16-row tiles
def test_no_row_layout_at_all(psx, n):
    import peasoup_amd.workloads as W
    w = workload(W, n)
    with pytest.raises(psx.PsxError, match="row-layout"):
        W.batch_search(w.search_args(), W.generate_host(w), w.dm_list(), None,
                       W.make_batch_opts(2, spectrum_layout=W.SPECTRUM_ROWS))
