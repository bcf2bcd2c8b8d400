"""Harmonic sums at the edges of a wave's 256 bins and of a workgroup's 1,024,
against the oracle."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nfolds", [1, 4, 5])
@pytest.mark.parametrize("nb", [255, 256, 257, 319, 1023, 1024, 1025, 1281])
def test_wave_and_group_edges(psx, orc, nfolds, nb):
    P = np.random.default_rng(nb).standard_normal(nb).astype(np.float32)
    d_P = psx.DeviceArray.from_numpy(P)
    folds = [psx.DeviceArray.from_numpy(np.full(nb + 1, -7, np.float32)) for _ in range(nfolds)]
    arr = (C.c_void_p * nfolds)(*[f.ptr for f in folds])
    psx.check(psx.lib().psx_harmonic_sum(d_P.ptr, arr, nfolds, nb, None))
    ref = orc.harmonic_sum(P, nfolds)
    for k in range(nfolds):
        got = folds[k].numpy()
        assert np.array_equal(got[:nb], ref[k]) and got[nb] == -7
