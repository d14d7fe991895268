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

pytestmark = pytest.mark.gpu


def _windows(P):
    run = P // 8
    return [(-run, run - 1), (-run - 1, 3), (2, run), (-2 * run, 2 * run - 1), (-2 * run - 1, 5), (-3, 2 * run),
            (run // 2, run // 2), (-run, -run), (P // 2, P // 2), (1 - P // 2, 1 - P // 2), (run + 3, P // 2),
            (1 - P // 2, -run - 5)]


@pytest.mark.parametrize("P,C", [(1024, 1), (1024, 3), (1024, 5), (2048, 1), (2048, 2), (2048, 3), (2048, 5),
                                 (3072, 1), (3072, 4), (3072, 7), (4096, 1), (4096, 3), (4096, 6), (4096, 7),
                                 (4096, 8), (5120, 1), (5120, 2), (6144, 1), (6144, 2), (8192, 1), (8192, 4)])
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
