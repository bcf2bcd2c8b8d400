"""Rows staged for a group of DM trials hold every stretch its trials read:
the host rule against the delays themselves, up to the longest ones."""
import os
import shutil
import subprocess

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
f32 = np.float32
PROGRAM = r'''
#include <cstdio>
#include <vector>
#include "dedisp_pitch.hpp"
int main() {  // lines: ndm per tmax, then the DMs
  unsigned n, per;
  float tmax;
  while (std::scanf("%u %u %f", &n, &per, &tmax) == 3) {
    std::vector<float> dm(n);
    for (float& d : dm)
      if (std::scanf("%f", &d) != 1) return 1;
    std::printf("%u\n", psx::staged_pitch(dm.data(), n, per, tmax));
  }
}
'''


@pytest.fixture(scope="module")
def pitches(tmp_path_factory):
    cxx = shutil.which("g++")
    if not cxx:
        pytest.skip("no g++")
    d = tmp_path_factory.mktemp("pitch")
    (d / "p.cpp").write_text(PROGRAM)
    subprocess.run([cxx, "-std=c++17", "-O1", "-I", os.path.join(ROOT, "peasoup_amd", "csrc"), str(d / "p.cpp"), "-o",
                    str(d / "p")], check=True)

    def run(lists):
        text = "".join("%d %d %.9g\n%s\n" % (len(dm), per, tab, " ".join("%.9g" % x for x in dm))
                       for dm, per, tab in lists)
        out = subprocess.run([str(d / "p")], input=text, capture_output=True, text=True, check=True).stdout
        return [int(x) for x in out.split()]

    return run


@pytest.mark.parametrize("log_delay", [4, 10, 15, 20, 23, 24, 25, 26, 27, 28, 29, 30])
def test_stretches_fit(pitches, log_delay):
    rng = np.random.default_rng(log_delay)
    lists = []
    for _ in range(3000):
        per = int(rng.choice([16, 32]))
        tab = f32(rng.uniform(1, 2) * 2.0 ** rng.integers(0, 8))
        first = 2.0 ** log_delay * rng.uniform(1, 1.9) / tab
        dm = np.sort((first + np.linspace(0, rng.uniform(0, 900) / tab, rng.integers(3, 50))).astype(f32))
        lists.append((dm, per, tab))
    for (dm, per, tab), pitch in zip(lists, pitches(lists)):
        delay = np.rint(dm * tab).astype(np.int64)
        for g in range(0, dm.size, per):
            d = delay[g:g + per]
            # a lane's last dword of the group's last trial: 255 past its first
            assert int(d[-1] - d[0]) // 4 + 256 <= pitch, (dm, tab)


@pytest.mark.gpu
@pytest.mark.parametrize("delay,spread", [
    (1017, 1016), (1017, 1000),  # the widest spread staged (512 dwords)
    (5000, 1000), ((1 << 24) + 3, 1000), ((1 << 28) + 77, 960),
])
def test_long_delays(psx, delay, spread):
    """Two channels, the second delayed by up to `delay` samples."""
    import peasoup_amd.sigproc as sigproc
    dt, f0, df = f32(0.000256), f32(1500.0), f32(-150.0)
    tab = sigproc.delay_table(2, dt, f0, df)
    ndm = 16
    top = delay / float(tab[1])
    dms = np.linspace(max(0.0, top - spread / float(tab[1])), top, ndm).astype(f32)
    lag = np.rint(dms * tab[1]).astype(np.int64)
    nout = 2500
    n = int(lag[-1]) + nout
    x = np.empty((n, 2), np.uint8)
    x[:, 0] = np.resize(np.random.default_rng(delay).integers(0, 256, 65521, dtype=np.uint8), n)
    x[:, 1] = np.resize(np.random.default_rng(delay + 1).integers(0, 256, 65519, dtype=np.uint8), n)
    d_in = psx.DeviceArray.from_numpy(x)
    d_out = psx.DeviceArray((ndm, nout))
    work = psx.DeviceArray(int(psx.lib().psx_dedisp_work_bytes(n, 2, ndm)), np.uint8)
    psx.check(psx.lib().psx_dedisperse(d_in.ptr, n, 2, 8, dms.ctypes.data, ndm, None, dt, f0, df, d_out.ptr, nout,
                                       work.ptr, None))
    got = d_out.numpy()
    for d in range(ndm):
        want = (x[:nout, 0].astype(f32) + x[lag[d]:lag[d] + nout, 1]) / f32(255 * 2)
        assert np.array_equal(got[d], want), d
