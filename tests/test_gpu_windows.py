"""Lag windows of the FFT form on every workgroup shape of the pair kernel.

The pair kernel is built for windows inside one or two runs of P/8 lags on
either side of lag 0, for any window, and for the full lag range, each in
several workgroup shapes chosen by the channel count.  Windows that end on,
just before and just after a run's edge, one-lag windows at the ends of the
lag range and one-sided windows, on traces long enough that the circular wrap
matters, against FP64 direct sums.

Bars, as for the other FFT-form tests: coefficients within 1e-5, lags equal
wherever the FP64 gap of the two best lags is at least 1e-12."""
import ctypes

import numpy as np
import pytest

from seismic_amd import engine, synth
from seismic_amd.device import DeviceArray, synchronize

pytestmark = pytest.mark.gpu


def _ncc_f64(x, L, P, lo, hi, demean):
    """Every pair's coefficients over the window, FP64 FFTs of period P: norms
    (and means) of the first L samples, lags circular mod P."""
    y = np.zeros(x.shape[:2] + (P,))
    y[..., :x.shape[-1]] = x
    if demean:
        y[..., :L] = (y[..., :L] - y[..., :L].mean(-1, keepdims=True)).astype(np.float32)
    nr = np.sqrt((y[..., :L] ** 2).sum(-1, keepdims=True))
    f = np.fft.rfft(np.divide(y, nr, out=np.zeros_like(y), where=nr > 0))
    i, j = np.triu_indices(x.shape[0])
    c = np.fft.irfft((f[i] * np.conj(f[j])).mean(1), n=P)
    return c[:, np.arange(lo, hi + 1) % P]


def _windows(P):
    run = P // 8
    return [(-run, run - 1), (-run - 1, 3), (2, run), (-2 * run, 2 * run - 1), (-2 * run - 1, 5), (-3, 2 * run),
            (run // 2, run // 2), (-run, -run), (P // 2, P // 2), (1 - P // 2, 1 - P // 2), (run + 3, P // 2),
            (1 - P // 2, -run - 5)]


@pytest.mark.parametrize("P,C", [(1024, 1), (1024, 3), (1024, 5), (2048, 1), (2048, 2), (2048, 3), (2048, 5),
                                 (3072, 1), (3072, 4), (3072, 7), (4096, 1), (4096, 3), (4096, 6), (4096, 7),
                                 (4096, 8), (5120, 1), (5120, 2), (5120, 6), (6144, 1), (6144, 2), (6144, 8), (8192, 1),
                                 (8192, 4), (8192, 8)])
def test_windows_at_run_edges(oracle, P, C):
    n, L = 5, P - 200
    ev, _ = synth.make_events(n, C, L, seed=P + C)
    pi, pj = oracle.packed_pairs(n)
    for lo, hi in _windows(P):
        print(f"case window P={P} C={C} [{lo}, {hi}]", flush=True)
        vp, lp, vn, ln = engine.allpairs_host(ev, P, lo, hi)
        ref = oracle.pairs_f64(ev, pi, pj, lo, hi, P=P, circular=True)
        assert np.abs(vp - ref["pos"]).max() <= 1e-5 and np.abs(vn - ref["neg"]).max() <= 1e-5
        sp, sn = ref["gap_pos"] >= 1e-12, ref["gap_neg"] >= 1e-12
        assert np.array_equal(lp[sp], ref["lag_pos"][sp]) and np.array_equal(ln[sn], ref["lag_neg"][sn])


@pytest.mark.parametrize("n", [1, 2, 7, 8, 9, 17, 31, 33, 64, 65, 130, 257, 420])
def test_small_jobs_every_column_chunk(oracle, n):
    """Event counts at and around the multiples of 8, 16, 32 and 64 columns
    that a small job's work items take: every pair of the triangle."""
    C, L, P, lo, hi = 1 + n % 3, 300, 1024, -20, 23
    ev, _ = synth.make_events(n, C, L, seed=500 + n)
    print(f"case small job N={n} C={C}", flush=True)
    vp, lp, vn, ln = engine.allpairs_host(ev, P, lo, hi)
    pi, pj = oracle.packed_pairs(n)
    ref = oracle.pairs_f64(ev, pi, pj, lo, hi, P=P, circular=True)
    assert np.abs(vp - ref["pos"]).max() <= 1e-5 and np.abs(vn - ref["neg"]).max() <= 1e-5
    sp, sn = ref["gap_pos"] >= 1e-12, ref["gap_neg"] >= 1e-12
    assert np.array_equal(lp[sp], ref["lag_pos"][sp]) and np.array_equal(ln[sn], ref["lag_neg"][sn])


@pytest.mark.parametrize("P,L,in_len,lo,hi,C,demean", [
    (4096, 2048, 2048, -512, 512, 3, False),    # period 3072 serves the window
    (4096, 2048, 2048, -1024, 1024, 1, False),  # L + max |lag| = 3072 exactly
    (4096, 2048, 2048, -1025, 1000, 1, False),  # one more: 4096
    (8192, 4096, 3000, -512, 512, 1, False),    # rows shorter than L
    (4096, 2000, 2300, -512, 512, 2, False),    # rows longer than L, still below 3072
    (4096, 1500, 4000, -400, 400, 1, False),    # rows too long for the smaller period: wrap at 4096
    (2048, 1000, 2048, -20, 20, 1, False),      # rows of P samples
    (3072, 1500, 1500, -1499, 1499, 2, False),  # every overlapping lag: scanned unmasked
    (3072, 1500, 1500, -1499, 1500, 2, True),
    (4096, 1200, 700, -100, 100, 1, True),      # demeaned up to L, beyond the rows
    (4096, 1200, 700, -1199, 1199, 1, True),
    (4096, 100, 100, 50, 1500, 1, False),       # window past the traces: half a period must hold it
    (8192, 300, 300, -299, 299, 5, False),
])
def test_period_follows_rows_and_window(P, L, in_len, lo, hi, C, demean):
    """Executes run at the smallest period that gives the window's lags of the
    circular correlation mod P, and scan every lag where the window covers all
    overlaps.  A silent event and events of a single sample among the others:
    most of their values are exact zeros, which must come out as (0, lag 0)."""
    x, _ = synth.make_events(12, C, max(in_len, 90), seed=P + L + hi)
    x = x[..., :in_len].copy()
    if demean:
        x += np.float32(0.5)
    x[3] = 0.0
    x[4:6] = 0.0
    x[4, :, in_len // 3] = 2.0
    x[5, :, in_len // 2] = -1.0
    print(f"case period P={P} L={L} in_len={in_len} [{lo}, {hi}] C={C} demean={demean}", flush=True)
    plan = engine.AllPairsPlan(12, C, L, P, lo, hi, demean=demean)
    out = plan.execute(DeviceArray.from_numpy(x))
    synchronize()
    vp, lp, vn, ln = [o.numpy() for o in out]
    plan.close()
    c = _ncc_f64(x, L, P, lo, hi, demean)
    for v, lag, sign in ((vp, lp, 1.0), (-vn, ln, -1.0)):
        w = np.sort(sign * c, axis=-1)
        best, gap = w[:, -1], w[:, -1] - w[:, -2]
        assert np.abs(v - np.maximum(best, 0.0)).max() <= 1e-5
        none = best <= 1e-12  # FP64 rounding around an exact zero
        assert not v[none].any() and not lag[none].any()
        sure = ~none & (gap >= 1e-12)
        assert np.array_equal(lag[sure], lo + np.argmax(sign * c, axis=-1)[sure])


@pytest.mark.parametrize("P,L,in_len,lo,hi,C,demean", [
    (8192, 4096, 4096, -50, 50, 1, False),     # segments of 924 samples at period 1024
    (8192, 4095, 4095, -50, 50, 1, True),
    (8192, 4096, 4096, -512, 512, 1, False),   # 1024 samples at 2048
    (8192, 4096, 4096, -511, 500, 2, True),
    (8192, 4095, 3000, -50, 50, 1, False),     # rows shorter than L: fewer segments
    (8192, 4095, 3000, -50, 50, 1, True),      # demeaned up to L, beyond the rows
    (8192, 4000, 4300, -20, 20, 1, True),      # rows longer than L, still within the segments
    (8192, 4096, 8192, -50, 50, 1, False),     # rows of P samples: whole rows, wrap at 8192
    (8192, 4096, 700, -50, 50, 1, False),      # rows of less than one segment
    (8192, 4000, 4000, 100, 400, 1, False),    # one-sided windows
    (8192, 4000, 4000, -400, -100, 1, False),
    (8192, 4000, 4000, -1023, 1024, 1, False),
    (4096, 2048, 2048, -100, 100, 1, False),
    (4096, 1999, 1999, -37, 36, 3, True),
    (4096, 2049, 2049, 0, 1, 2, False),
    (2048, 1100, 1100, 5, 6, 4, False),
    (3072, 2900, 2900, -1, 170, 2, False),
])
def test_rows_in_segments(P, L, in_len, lo, hi, C, demean):
    """Windows far shorter than the traces: the rows are cut in segments at a
    shorter period, whose products are summed before one transform."""
    test_period_follows_rows_and_window(P, L, in_len, lo, hi, C, demean)


@pytest.mark.parametrize("demean", [False, True])
def test_segments_host_call_and_no_allocation(demean):
    """A job big enough for event bands, and the entry point without
    allocations, against the plan's own execute: bitwise equal."""
    n, C, L, P, lo, hi = 1100, 1, 3001, 8192, -60, 45
    x, _ = synth.make_events(n, C, L, seed=9)
    x += np.float32(0.25 * demean)
    d = DeviceArray.from_numpy(x)
    plan = engine.AllPairsPlan(n, C, L, P, lo, hi, demean=demean)
    print(f"case segments host and noalloc demean={demean}", flush=True)
    out = plan.execute(d)
    synchronize()
    want = [o.numpy() for o in out]
    host = engine.allpairs_host(x, P, lo, hi, demean=demean)
    for o in out:
        o.zero_()
    rc = plan.lib.sxc_plan_execute_noalloc(ctypes.byref(plan.desc), ctypes.c_void_p(d.ptr), L, L,
                                           *(ctypes.c_void_p(o.ptr) for o in out), ctypes.c_void_p(0))
    assert rc == 0
    synchronize()
    for w, h, o in zip(want, host, out):
        assert np.array_equal(w, h) and np.array_equal(w, o.numpy())
    plan.close()


@pytest.mark.parametrize("P", [5120, 6144, 8192])
@pytest.mark.parametrize("n", [1, 3, 4, 5, 11, 32, 66])
def test_small_jobs_of_four_wave_workgroups(P, n):
    """One channel at the periods whose workgroups have four waves: items of 4
    columns in the smallest jobs."""
    L, lo, hi = P // 2 + 100, -P // 2 + 1, P // 2
    ev, _ = synth.make_events(n, 1, L, seed=P + n)
    print(f"case four-wave job N={n} P={P}", flush=True)
    vp, lp, vn, ln = engine.allpairs_host(ev, P, lo, hi)
    c = _ncc_f64(ev, L, P, lo, hi, False)
    for v, lag, sign in ((vp, lp, 1.0), (-vn, ln, -1.0)):
        w = np.partition(sign * c, -2, axis=-1)[:, -2:]  # the two best
        assert np.abs(v - np.maximum(w[:, 1], 0.0)).max() <= 1e-5
        sure = (w[:, 1] > 1e-12) & (w[:, 1] - w[:, 0] >= 1e-12)
        assert np.array_equal(lag[sure], lo + np.argmax(sign * c, axis=-1)[sure])


def test_loud_rows_past_the_trace_length_stay_in_the_window():
    """Rows longer than L with loud samples past it: coefficients far above 1,
    whose rounding at lags outside the window is no near tie of 0.  Positive
    traces have no negative side; no reported lag may leave the window."""
    n, L, in_len, P = 12, 500, 1400, 3072
    lo, hi = 1 - in_len, in_len - 1
    x = np.random.default_rng(3).uniform(1.0, 2.0, (n, 1, in_len)).astype(np.float32)
    x[..., :L] *= np.float32(0.01)
    print(f"case loud rows P={P} L={L} in_len={in_len} [{lo}, {hi}]", flush=True)
    plan = engine.AllPairsPlan(n, 1, L, P, lo, hi)
    out = plan.execute(DeviceArray.from_numpy(x))
    synchronize()
    vp, lp, vn, ln = [o.numpy() for o in out]
    plan.close()
    c = _ncc_f64(x, L, P, lo, hi, False)
    assert (c > 0.05).all() and np.abs(vp / c.max(-1) - 1.0).max() <= 1e-5
    assert ((lp >= lo) & (lp <= hi)).all()
    assert not vn.any() and not ln.any()
