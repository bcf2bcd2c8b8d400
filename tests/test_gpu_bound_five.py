"""Five folds: the pairs whose bound crosses are first summed again from the
bins' own bounds.  The candidates are the exact pass's at thresholds where few
pairs of a row cross (so that they take this way), in both spectrum layouts."""
import pytest

from test_gpu_bound import both_forms, same

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("thr", [5.5, 6.0, 7.0])
@pytest.mark.parametrize("n", [1 << 17, 3 << 18])
@pytest.mark.parametrize("layout", ["natural", "rows"])
def test_five_folds_bound_equals_exact(psx, thr, n, layout):
    import peasoup_amd.workloads as W
    w = W.Workload("five", 2, n, 64e-6, 0x5EB500, 5.0, -20.0, 20.0, nharmonics=5, min_snr=thr,
                   injections=[W.Injection(0, 0.0123, 5.0, 20.0, 0.03), W.Injection(1, 0.301, 0.0, 15.0, 0.02)])
    series = W.generate_host(w)
    accs = W.accel_list(w.size, w.tsamp, w.acc_lo, w.acc_hi)[:13]
    kw = {"decomp": [(256, 16), (n // 512, 8 if n // 512 > 256 else 16)],
          "spectrum_layout": W.SPECTRUM_NATURAL if layout == "natural" else W.SPECTRUM_ROWS}
    bound, exact = both_forms(W, w, series, accs, 8, **kw)
    assert len(exact) > 0
    assert same(bound, exact) and len(bound) == len(exact)
