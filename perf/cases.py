"""Cases by which the speed of the search core is followed.

Each case is one pass through the public entry points as a user's program
calls them: whole searches (batched, served, plain Worker), the plain
per-stage chains below the drop-in transform classes, single FFT plans and
dedispersion.  ``listed()`` names the standing cases, ``draw(rng)`` gives
another one of the same ranges, ``prepare``/``run`` make the inputs and do
the pass, ``work`` counts what a pass cannot do without and ``exact`` gives
the per-stage results in 64 bits.
"""
import ctypes as C
import functools
import math

import numpy as np
import torch

import peasoup_amd as P
import peasoup_amd.sigproc as sigproc
import peasoup_amd.workloads as W
from peasoup_amd import tuning
from peasoup_amd.serve import Server

CAND_ROWS = 1 << 16  # candidate records a search case returns (unused ones zero)
PEAK_ROWS = 8192  # above-threshold bins a plain trial returns per spectrum
# a short observatory zap list (mains and its harmonics), Hz and half-width
ZAPS = ((50.0, 0.05), (100.0, 0.05), (150.0, 0.08), (200.0, 0.1))
SERVE_SIZES = {"short": ((20, 32), (20, 16), (21, 16)), "mixed": ((20, 24), (21, 16), (22, 8), (23, 4))}


def listed():
    return [
        # Smallest search: 8 DM trials of 2^17 samples, series still in host
        # memory (the CPU-sized benchmark configuration); launches and host
        # round trips count.
        {"name": "search_2p17_host", "kind": "search", "n": 1 << 17, "nreal": 1 << 17, "ndm": 8, "tsamp": 64e-6,
         "acc": 50.0, "nharm": 4, "zap": False, "host": True},
        # A short beam of the serving mix: 64 DMs of 2^20 samples, +-200 m/s^2
        # (a handful of accelerations per DM).
        {"name": "search_2p20", "kind": "search", "n": 1 << 20, "nreal": 1 << 20, "ndm": 64, "tsamp": 64e-6,
         "acc": 200.0, "nharm": 4, "zap": False, "host": False},
        # A segmented search of uneven length: 3*2^21, 90% real samples (zero
        # padded), with a zap list.
        {"name": "search_3x2p21_padded", "kind": "search", "n": 3 << 21, "nreal": int(0.9 * (3 << 21)), "ndm": 16,
         "tsamp": 76e-6, "acc": 50.0, "nharm": 4, "zap": True, "host": False},
        # The headline workload (2^23 samples, +-100 m/s^2, 127 accelerations
        # per DM) on 16 of its DM trials.
        {"name": "search_2p23", "kind": "search", "n": 1 << 23, "nreal": 1 << 23, "ndm": 16, "tsamp": 76e-6,
         "acc": 100.0, "nharm": 4, "zap": False, "host": False},
        # Long segment: one DM of 2^26 samples over a narrow acceleration range.
        {"name": "search_2p26", "kind": "search", "n": 1 << 26, "nreal": 1 << 26, "ndm": 1, "tsamp": 64e-6,
         "acc": 4.0, "nharm": 4, "zap": False, "host": False},
        # Requests of four lengths submitted together to the server.
        {"name": "serve_mixed", "kind": "serve", "mix": "mixed", "tsamp": 64e-6, "acc": 50.0},
        # The drop-in path: the Worker's sequence, one library call per
        # reference call, host series.
        {"name": "worker_2p20", "kind": "worker", "n": 1 << 20, "nreal": 1000003, "ndm": 4, "tsamp": 64e-6,
         "acc": 200.0, "nharm": 4},
        # One plain acceleration trial through the C ABI: resample, R2C,
        # interbin, normalise, four folds, peaks of all five spectra.
        {"name": "trial_2p23", "kind": "trial", "n": 1 << 23, "acc": 50.0, "tsamp": 76e-6, "nharm": 4},
        # One plain DM prologue through the C ABI: baseline, R2C, amplitude,
        # running median, deredden, interbin, statistics, C2R.
        {"name": "prologue_2p22", "kind": "prologue", "n": 1 << 22, "nreal": 4000001, "tsamp": 64e-6, "zap": True},
        # A plain batched R2C of a radix-3 length.
        {"name": "fft_r2c_3x2p17_b8", "kind": "fft", "n": 3 << 17, "batch": 8, "inverse": False},
        # Dedispersion of a small 2-bit filterbank (the tutorial file's
        # shape: 64 channels, 187520 samples, 59 DM trials).
        {"name": "dedisp_2bit_64ch", "kind": "dedisperse", "nbits": 2, "nchans": 64, "nsamps": 187520, "ndm": 59,
         "tsamp": 320e-6, "f0": 1510.0, "bw": 69.76, "dm_end": 253.2, "masked": 0},
        # Dedispersion of an 8-bit survey gulp, some channels masked.
        {"name": "dedisp_8bit_1024ch", "kind": "dedisperse", "nbits": 8, "nchans": 1024, "nsamps": (1 << 19) + 321,
         "ndm": 128, "tsamp": 64e-6, "f0": 1510.0, "bw": 400.0, "dm_end": 120.0, "masked": 37},
    ]


def _length(rng, lo, hi):
    """A length 2^k or 3*2^k with lo <= k <= hi (k the power of two below it)."""
    k = rng.randint(lo, hi)
    return 3 << (k - 1) if k < hi and rng.random() < 0.35 else 1 << k


def draw(rng):
    kind = rng.choice(["search", "search", "search", "serve", "worker", "trial", "prologue", "fft", "dedisperse",
                       "dedisperse"])
    tsamp = rng.choice([64e-6, 76e-6])
    if kind == "search":
        n = _length(rng, 17, 24)
        ndm = rng.randint(1, max(1, min(64, (1 << 26) // n)))
        frac = 1.0 if rng.random() < 0.5 else rng.uniform(0.55, 1.0)
        # accelerations: as wide as the range, and no more trials than the listed largest
        acc = rng.choice([20.0, 50.0, 100.0, 200.0])
        while acc > 1.0 and n * ndm * W.accel_list(n, tsamp, -acc, acc).size > 1.2e10:
            acc /= 2.0
        return {"kind": kind, "n": n, "nreal": int(frac * n), "ndm": ndm, "tsamp": tsamp, "acc": acc,
                "nharm": rng.randint(1, 5), "zap": rng.random() < 0.3, "host": rng.random() < 0.25}
    if kind == "serve":
        return {"kind": kind, "mix": rng.choice(sorted(SERVE_SIZES)), "tsamp": tsamp,
                "acc": round(rng.uniform(20.0, 60.0), 3)}
    if kind == "worker":
        n = _length(rng, 17, 22)
        acc = round(rng.uniform(20.0, 200.0), 2)
        while n * W.accel_list(n, tsamp, -acc, acc).size > 5e7:
            acc = round(acc / 2.0, 3)
        return {"kind": kind, "n": n, "nreal": int(rng.uniform(0.55, 1.0) * n), "ndm": rng.randint(1, 4),
                "tsamp": tsamp, "acc": acc, "nharm": rng.randint(1, 5)}
    if kind == "trial":
        return {"kind": kind, "n": _length(rng, 17, 24), "acc": round(rng.uniform(-200.0, 200.0), 3), "tsamp": tsamp,
                "nharm": rng.randint(1, 5)}
    if kind == "prologue":
        n = _length(rng, 17, 24)
        return {"kind": kind, "n": n, "nreal": int(rng.uniform(0.55, 1.0) * n), "tsamp": tsamp,
                "zap": rng.random() < 0.5}
    if kind == "fft":
        n = _length(rng, 12, 23)
        return {"kind": kind, "n": n, "batch": rng.randint(1, max(1, min(64, (1 << 24) // n))),
                "inverse": rng.random() < 0.5}
    nbits = rng.choice([1, 2, 4, 8])
    nchans = 8 * rng.randint(4, 128)
    ndm = rng.randint(3, 160)
    nsamps = int(math.exp(rng.uniform(math.log(30000), math.log(1 << 19))))
    bw = rng.uniform(60.0, 400.0)
    # the delay across the band takes at most a third of the samples
    per_dm = 4.15e3 / tsamp * (1.0 / (1510.0 - bw) ** 2 - 1.0 / 1510.0 ** 2)
    dm_end = round(rng.uniform(0.2, 1.0) * min(300.0, nsamps / 3.0 / per_dm), 3)
    return {"kind": kind, "nbits": nbits, "nchans": nchans, "nsamps": nsamps, "ndm": ndm, "tsamp": tsamp,
            "f0": 1510.0, "bw": round(bw, 3), "dm_end": dm_end, "masked": rng.randint(0, nchans // 16)}


# ------------------------------------------------------------------ inputs
@functools.lru_cache(maxsize=None)
def _search_args(n, tsamp, acc, nharm, zap):
    """The search settings of a program: one object for all its segments."""
    return W.make_search_args(n, tsamp, acc_start=-acc, acc_end=acc, nharmonics=nharm, birdies=ZAPS if zap else None)


@functools.lru_cache(maxsize=None)
def _device_name():
    return P.device_info(0)["name"]


def _workload(case, seed, n, nreal, ndm, acc=50.0):
    """N(0,1) noise with red noise, and one or two accelerated pulsars."""
    w = W.Workload("case", ndm, n, case["tsamp"], int(seed), 5.0, nsamps=nreal)
    rng = np.random.default_rng(int(seed))
    for t in rng.choice(ndm, min(ndm, 2), replace=False):
        w.injections.append(W.Injection(int(t), float(rng.uniform(2e-3, 0.1)), float(rng.uniform(-0.8, 0.8) * acc),
                                        float(rng.uniform(12, 40)), float(rng.random())))
    return w


def _host_series(w):
    return W.generate_host(w)


def _series_tensor(case, seed, n, nreal):
    """One series in a torch tensor of n samples (the last n - nreal zero)."""
    x = torch.zeros(n, dtype=torch.float32, device="cuda")
    torch.cuda.synchronize()
    w = _workload(case, seed, n, nreal, 1, 20.0)
    W.SeriesGenerator(nreal).generate(x.data_ptr(), nreal, w.tsamp, w.seed, 0, w.red_amp, w.injections)
    P.synchronize()
    return x


def _bytes(n):
    return torch.empty(max(int(n), 1), dtype=torch.uint8, device="cuda")


def _dedisp_setup(case):
    dms = np.linspace(0.0, case["dm_end"], case["ndm"]).astype(np.float32)
    df = np.float32(-case["bw"] / case["nchans"])
    dt, f0 = np.float32(case["tsamp"]), np.float32(case["f0"])
    table = sigproc.delay_table(case["nchans"], dt, f0, df)
    nout = case["nsamps"] - int(P.lib().psx_dedisp_max_delay(dms.ctypes.data, dms.size, table.ctypes.data, table.size))
    mask = None
    if case["masked"]:
        mask = np.ones(case["nchans"], np.int32)
        mask[np.random.default_rng(7).choice(case["nchans"], case["masked"], replace=False)] = 0
    return dms, dt, f0, df, table, nout, mask


def prepare(case, seed):
    k = case["kind"]
    if k in ("search", "worker"):
        w = _workload(case, seed, case["n"], case["nreal"], case["ndm"], case["acc"])
        args = _search_args(case["n"], case["tsamp"], case["acc"], case["nharm"], case.get("zap", False))
        st = {"kind": k, "args": args, "dms": w.dm_list(), "nsamps": case["nreal"]}
        if k == "worker" or case["host"]:
            st["series"] = _host_series(w)
        else:
            st["series"] = W.generate_device(w)
            P.synchronize()
        if k == "search":
            tuned = tuning.lookup(case["n"], _device_name())
            st["opts"] = W.make_batch_opts(tuned.get("batch", 0), decomp=tuned.get("decomp"), keep_engine=True)
        return st
    if k == "serve":
        reqs = []
        for j, (lg, ndm) in enumerate(SERVE_SIZES[case["mix"]]):
            n = 1 << lg
            w = _workload(case, seed * 16 + j, n, n, ndm, case["acc"])
            reqs.append((_search_args(n, case["tsamp"], case["acc"], 4, False), W.generate_device(w), w.dm_list(), n))
        P.synchronize()
        return {"kind": k, "server": _ClosedServer(100e9, batch=64, schedules=tuning.table(_device_name())),
                "requests": reqs}
    if k == "trial":
        n, nb = case["n"], case["n"] // 2 + 1
        st = {"kind": k, "n": n, "nb": nb, "acc": case["acc"], "tsamp": case["tsamp"],
              "x": _series_tensor(case, seed, n, n), "r": torch.empty(n, dtype=torch.float32, device="cuda"),
              "X": torch.empty(nb, dtype=torch.complex64, device="cuda"),
              "P": torch.empty(nb, dtype=torch.float32, device="cuda"),
              "folds": [torch.empty(nb, dtype=torch.float32, device="cuda") for _ in range(case["nharm"])],
              "idx": [torch.zeros(PEAK_ROWS, dtype=torch.int32, device="cuda") for _ in range(case["nharm"] + 1)],
              "snr": [torch.zeros(PEAK_ROWS, dtype=torch.float32, device="cuda") for _ in range(case["nharm"] + 1)],
              "count": torch.zeros(case["nharm"] + 1, dtype=torch.int32, device="cuda"),
              "work": _bytes(P.lib().psx_find_peaks_work_bytes(nb)), "plan": P.FFTPlan(n)}
        st["fold_ptrs"] = (C.c_void_p * case["nharm"])(*[f.data_ptr() for f in st["folds"]])
        # the statistics the DM's prologue left; white enough above 1 Hz
        red = _bytes(P.lib().psx_reduce_work_bytes())
        torch.cuda.synchronize()
        mean, rms = C.c_float(), C.c_float()
        st["plan"].execute(st["x"].data_ptr(), st["X"].data_ptr())
        P.check(P.lib().psx_form_interbin(st["X"].data_ptr(), st["P"].data_ptr(), nb, None))
        P.check(P.lib().psx_mean_rms(st["P"].data_ptr(), nb, min(nb // 2, int(n * case["tsamp"])), C.byref(mean),
                                     C.byref(rms), red.data_ptr(), None))
        st["mean"] = mean.value
        st["std"] = math.sqrt(rms.value ** 2 - mean.value ** 2)
        return st
    if k == "prologue":
        n, nb = case["n"], case["n"] // 2 + 1
        lib = P.lib()
        st = {"kind": k, "n": n, "nb": nb, "nreal": case["nreal"], "bin_width": 1.0 / (n * case["tsamp"]),
              "raw": _series_tensor(case, seed, case["nreal"], case["nreal"]),
              "tim": torch.empty(n, dtype=torch.float32, device="cuda"),
              "X": torch.empty(nb, dtype=torch.complex64, device="cuda"),
              "A": torch.empty(nb, dtype=torch.float32, device="cuda"),
              "median": torch.empty(nb, dtype=torch.float32, device="cuda"),
              "med_work": torch.empty(int(lib.psx_deredden_work_floats(nb)), dtype=torch.float32, device="cuda"),
              "work": _bytes(lib.psx_reduce_work_bytes()), "zaps": None,
              "r2c": P.FFTPlan(n), "c2r": P.FFTPlan(n, P.PSX_FFT_C2R)}
        # an offset that the baseline removal takes out again
        st["raw"] += 0.25 + 0.5 * (seed % 7) / 7.0
        if case["zap"]:
            z = torch.tensor(ZAPS, dtype=torch.float32, device="cuda").t().contiguous()
            st["zaps"] = z
        torch.cuda.synchronize()
        return st
    if k == "fft":
        n, b = case["n"], case["batch"]
        g = torch.Generator(device="cuda").manual_seed(int(seed))
        if case["inverse"]:
            x = torch.randn(b, n // 2 + 1, 2, generator=g, device="cuda")
            x[:, 0, 1] = x[:, -1, 1] = 0.0  # the spectrum of a real series
            x = torch.view_as_complex(x)
            out = torch.empty(b, n, dtype=torch.float32, device="cuda")
        else:
            x = torch.randn(b, n, generator=g, device="cuda")
            out = torch.empty(b, n // 2 + 1, dtype=torch.complex64, device="cuda")
        torch.cuda.synchronize()
        return {"kind": k, "x": x, "out": out,
                "plan": P.FFTPlan(n, P.PSX_FFT_C2R if case["inverse"] else P.PSX_FFT_R2C, b)}
    if k == "dedisperse":
        dms, dt, f0, df, _, nout, mask = _dedisp_setup(case)
        g = torch.Generator(device="cuda").manual_seed(int(seed))
        size = case["nsamps"] * case["nchans"] * case["nbits"] // 8
        if case["nbits"] == 8:  # radiometer noise about the digitiser's middle
            packed = (torch.randn(size, generator=g, device="cuda") * 20.0 + 96.0).clamp_(0, 255).to(torch.uint8)
        else:
            packed = torch.randint(0, 256, (size,), generator=g, device="cuda", dtype=torch.uint8)
        torch.cuda.synchronize()
        return {"kind": k, "packed": packed, "nsamps": case["nsamps"], "nchans": case["nchans"],
                "nbits": case["nbits"], "dms": dms, "dt": dt, "f0": f0, "df": df, "mask": mask, "nout": nout,
                "out": torch.empty(case["ndm"], nout, dtype=torch.float32, device="cuda"),
                "work": _bytes(P.lib().psx_dedisp_work_bytes(case["nsamps"], case["nchans"], case["ndm"]))}
    raise KeyError(k)


class _ClosedServer(Server):
    """A server that shuts down with the program part that holds it."""

    def __del__(self):
        self.close()


# -------------------------------------------------------------------- pass
def _records(forest):
    """A candidate forest as plain columns of CAND_ROWS records."""
    out = np.zeros(CAND_ROWS, W.CAND_DTYPE)
    m = min(len(forest), CAND_ROWS)
    out[:m] = forest[:m]
    cols = {f: out[f] for f in ("dm", "dm_idx", "acc", "nh", "snr", "freq", "nassoc")}
    cols["count"] = len(forest)
    return cols


def run(state):
    k = state["kind"]
    lib = P.lib()
    if k == "search":
        forest, _ = W.batch_search(state["args"], state["series"], state["dms"], None, state["opts"],
                                   nsamps=state["nsamps"], forest=True)
        return _records(forest)
    if k == "worker":
        forest, _ = W.worker_search(state["args"], state["series"], state["dms"], forest=True)
        return _records(forest)
    if k == "serve":
        srv = state["server"]
        ids = [srv.submit(args, d, dms, nsamps=n) for args, d, dms, n in state["requests"]]
        out = []
        for i in ids:
            st = srv.wait(i, timeout=120.0)
            if st["state"] != "done":
                raise RuntimeError("request failed: %s" % st)
            out.append(_records(srv.result(i, forest=True)))
        return out
    if k == "trial":
        n, nb, s = state["n"], state["nb"], None
        P.check(lib.psx_resample(state["x"].data_ptr(), state["r"].data_ptr(), n, state["acc"], state["tsamp"], s))
        state["plan"].execute(state["r"].data_ptr(), state["X"].data_ptr(), s)
        p = state["P"].data_ptr()
        P.check(lib.psx_form_interbin(state["X"].data_ptr(), p, nb, s))
        P.check(lib.psx_normalise(p, state["mean"], state["std"], nb, s))
        P.check(lib.psx_harmonic_sum(p, state["fold_ptrs"], len(state["folds"]), nb, s))
        lo = int(n * state["tsamp"])  # 1 Hz
        for j, spec in enumerate([state["P"]] + state["folds"]):
            P.check(lib.psx_find_peaks(spec.data_ptr(), min(lo << j, nb), nb, 7.0, state["idx"][j].data_ptr(),
                                       state["snr"][j].data_ptr(), PEAK_ROWS, state["count"][j:].data_ptr(),
                                       state["work"].data_ptr(), s))
        return {"resampled": state["r"], "fourier": state["X"], "spectrum": state["P"], "folds": state["folds"],
                "idx": state["idx"], "snr": state["snr"], "count": state["count"]}
    if k == "prologue":
        n, nb, nreal, s = state["n"], state["nb"], state["nreal"], None
        tim, x, a = state["tim"].data_ptr(), state["X"].data_ptr(), state["A"].data_ptr()
        work = state["work"].data_ptr()
        P.check(lib.psx_memcpy_d2d(tim, state["raw"].data_ptr(), 4 * nreal, s))
        P.check(lib.psx_remove_baseline(tim, nreal, work, s))
        P.check(lib.psx_fill(tim, nreal, n, 0.0, s))
        state["r2c"].execute(tim, x, s)
        P.check(lib.psx_form_amplitude(x, a, nb, s))
        P.check(lib.psx_deredden_median(a, nb, state["bin_width"], 0.05, 0.5, state["median"].data_ptr(),
                                        state["med_work"].data_ptr(), s))
        P.check(lib.psx_divide_c_by_f(x, state["median"].data_ptr(), nb, s))
        if state["zaps"] is not None:
            P.check(lib.psx_zap_birdies(x, state["zaps"][0].data_ptr(), state["zaps"][1].data_ptr(), len(ZAPS),
                                        state["bin_width"], nb, s))
        P.check(lib.psx_form_interbin(x, a, nb, s))
        mean, rms = C.c_float(), C.c_float()
        P.check(lib.psx_mean_rms(a, nb, 0, C.byref(mean), C.byref(rms), work, s))
        state["c2r"].execute(x, tim, s)
        return {"tim": state["tim"], "fourier": state["X"], "spectrum": state["A"], "median": state["median"],
                "mean": mean.value, "rms": rms.value}
    if k == "fft":
        state["plan"].execute(state["x"].data_ptr(), state["out"].data_ptr())
        return state["out"]
    mask = state["mask"]
    P.check(lib.psx_dedisperse(state["packed"].data_ptr(), state["nsamps"], state["nchans"], state["nbits"],
                               state["dms"].ctypes.data, state["dms"].size, None if mask is None else mask.ctypes.data,
                               state["dt"], state["f0"], state["df"], state["out"].data_ptr(), state["nout"],
                               state["work"].data_ptr(), None))
    return state["out"]


# -------------------------------------------------------------------- work
def _trial_flops(n, nharm):
    """Resampling index, real FFT, spectrum forming and folds of one trial."""
    nb = n // 2 + 1
    return 2.0 * n + 2.5 * n * math.log2(n) + 12.0 * nb + nb * (2.0 ** nharm + nharm)


def _prologue_flops(n):
    nb = n // 2 + 1
    return 3.0 * n + 2 * 2.5 * n * math.log2(n) + 40.0 * nb


def work(case):
    k = case["kind"]
    if k in ("search", "worker"):
        naccs = W.accel_list(case["n"], case["tsamp"], -case["acc"], case["acc"]).size
        return {"bytes": 4.0 * case["nreal"] * case["ndm"] + 32 * 100,
                "flops": case["ndm"] * (_prologue_flops(case["n"]) + naccs * _trial_flops(case["n"], case["nharm"]))}
    if k == "serve":
        b = f = 0.0
        for lg, ndm in SERVE_SIZES[case["mix"]]:
            n = 1 << lg
            naccs = W.accel_list(n, case["tsamp"], -case["acc"], case["acc"]).size
            b += 4.0 * n * ndm
            f += ndm * (_prologue_flops(n) + naccs * _trial_flops(n, 4))
        return {"bytes": b, "flops": f}
    if k == "trial":
        n, nb = case["n"], case["n"] // 2 + 1
        # series in; resampled series, Fourier series, spectrum and folds out
        return {"bytes": 8.0 * n + 8.0 * nb + 4.0 * nb * (1 + case["nharm"]), "flops": _trial_flops(n, case["nharm"])}
    if k == "prologue":
        n, nb = case["n"], case["n"] // 2 + 1
        return {"bytes": 4.0 * case["nreal"] + 4.0 * n + 8.0 * nb + 8.0 * nb, "flops": _prologue_flops(n)}
    if k == "fft":
        n = case["n"]
        return {"bytes": case["batch"] * (4.0 * n + 8.0 * (n // 2 + 1)), "flops": case["batch"] * 2.5 * n * math.log2(n)}
    _, _, _, _, _, nout, _ = _dedisp_setup(case)
    return {"bytes": case["nsamps"] * case["nchans"] * case["nbits"] / 8.0 + 4.0 * case["ndm"] * nout,
            "flops": 1.0 * case["ndm"] * nout * (case["nchans"] - case["masked"])}


# ------------------------------------------------------------------- exact
def _interbin64(x):
    d = x.clone()
    d[1:] -= x[:-1]
    return torch.sqrt(torch.maximum(x.abs() ** 2, 0.5 * d.abs() ** 2))


def _scrunch64(a):
    return a[:a.numel() // 5 * 5].reshape(-1, 5).median(dim=1).values


def _stretch64(m, lo, hi, count):
    """Bins [lo, hi) of m stretched to count bins (float32 positions, as the
    stretch is defined)."""
    step = np.float32(np.float32(m.numel() - 1) / np.float32(count - 1))
    x = torch.arange(lo, hi, dtype=torch.float32) * torch.tensor(step)
    j = x.to(torch.int64)
    fr = (x - j.to(torch.float32)).double()
    last = m.numel() - 1
    a, b = m[j.clamp(max=last)], m[(j + 1).clamp(max=last)]
    return torch.where(fr > 1e-5, a + fr * (b - a), a)


def exact(case, seed):
    k = case["kind"]
    if k == "fft":
        x = prepare(case, seed)["x"].cpu()
        if case["inverse"]:
            return torch.fft.irfft(x.to(torch.complex128), n=case["n"], norm="forward")
        return torch.fft.rfft(x.double())
    if k == "trial":
        st = prepare(case, seed)
        n, nb = st["n"], st["nb"]
        af = float(np.float32(np.float32(st["acc"]) * np.float32(st["tsamp"]))) / (2 * 299792458.0)
        i = torch.arange(n, dtype=torch.float64)
        j = torch.round(i * af * (i - float(n)) + i).to(torch.int64).clamp_(0, n - 1)
        r = st["x"].cpu()[j].double()
        x = torch.fft.rfft(r)
        p = (_interbin64(x) - float(np.float32(st["mean"]))) / float(np.float32(st["std"]))
        b = torch.arange(nb, dtype=torch.int64)
        folds, val = [], p.clone()
        for m in range(1, case["nharm"] + 1):
            for h in range(1, 1 << m, 2):
                val = val + p[(b * h + (1 << (m - 1))) >> m]
            folds.append(val * 2.0 ** (-0.5 * m))
        return {"resampled": r, "fourier": x, "spectrum": p, "folds": folds, "idx": None, "snr": None, "count": None}
    if k == "prologue":
        st = prepare(case, seed)
        n, nb, nreal, bw = st["n"], st["nb"], st["nreal"], st["bin_width"]
        raw = st["raw"].cpu().double()
        tim = torch.zeros(n, dtype=torch.float64)
        tim[:nreal] = raw - raw.mean()
        x = torch.fft.rfft(tim)
        m5 = _scrunch64(x.abs())
        m25 = _scrunch64(m5)
        m125 = _scrunch64(m25)
        f32 = np.float32
        pos5 = min(int(float(f32(0.05)) / bw), nb)
        pos25 = min(int(float(f32(0.5)) / bw), nb)
        med = torch.cat([_stretch64(m5, 0, pos5, nb), _stretch64(m25, pos5, pos25, nb),
                         _stretch64(m125, pos25, nb, nb)])
        x = x / med
        x[:5] = 0
        if case["zap"]:
            for f, w in ZAPS:
                lo = int(math.floor(f32(f32(f32(f) - f32(w)) / f32(bw))))
                hi = int(math.ceil(f32(f32(f32(f) + f32(w)) / f32(bw))))
                x[max(lo, 0):max(min(hi, nb - 1), 0)] = 1.0
        a = _interbin64(x)
        return {"tim": torch.fft.irfft(x, n=n, norm="forward"), "fourier": x, "spectrum": a, "median": med,
                "mean": float(a.mean()), "rms": float((a * a).mean().sqrt())}
    if k == "dedisperse":
        if case["ndm"] * case["nchans"] > 400000:
            return None
        st = prepare(case, seed)
        dms, _, _, _, table, nout, mask = _dedisp_setup(case)
        per, bits = 8 // case["nbits"], case["nbits"]
        rows = st["packed"].reshape(case["nsamps"], -1)
        out = torch.zeros(case["ndm"], nout, dtype=torch.float64, device="cuda")
        for c in range(case["nchans"]):
            if mask is not None and not mask[c]:
                continue
            v = ((rows[:, c // per] >> ((c % per) * bits)) & ((1 << bits) - 1)).double()
            for d in range(case["ndm"]):
                t = int(np.rint(dms[d] * table[c]))
                out[d] += v[t:t + nout]
        return out / (float((1 << bits) - 1) * case["nchans"])
    return None
