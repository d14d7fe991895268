"""Lag windows of the FFT form on every workgroup shape of the pair kernel.

The pair kernel is built for windows inside one or two runs of P/8 lags on
either side of lag 0, for any window, and for the full lag range, each in
several workgroup shapes chosen by the channel count.  Windows that end on,
just before and just after a run's edge, one-lag windows at the ends of the
lag range and one-sided windows, on traces long enough that the circular wrap
matters, against FP64 direct sums.

Bars, as for the other FFT-form tests: coefficients within 1e-5, lags equal
wherever the FP64 gap of the two best lags is at least 1e-12."""
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
