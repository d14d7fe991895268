"""The lag-window forms over the shapes of their pair kernel: windows of one
block of 32 lags, one lag fewer and more, one and several ranges of blocks
(whole and one block short), one-sided windows (whose ranges skip the samples
no lag of theirs uses), traces of odd lengths down to fewer samples than a
product takes, jobs small enough that several waves share a row's ranges and
large enough that a wave takes two rows.  Every pair against FP64 direct sums.

Bars as for the other lag-form tests: coefficients within 1e-5 (bf16x3) and
2e-3 (fp16), lags equal wherever the FP64 gap of the two best lags is at least
1e-12 (values above 1e-3)."""
import ctypes

import numpy as np
import pytest

from seismic_amd import engine, tiled
from seismic_amd.device import DeviceArray, synchronize

pytestmark = pytest.mark.gpu

FORMS = {"bf16x3": (engine.FORM_LAG_BF16X3, 1e-5), "fp16": (engine.FORM_LAG_FP16, 2e-3)}


@pytest.mark.parametrize("name", ["bf16x3", "fp16"])
@pytest.mark.parametrize("n,C,L,lo,hi", [
    (5, 1, 9, -8, 8), (5, 1, 40, -39, 39), (33, 2, 100, -15, 15), (34, 1, 333, 0, 31), (34, 1, 333, 1, 33),
    (34, 1, 333, -200, -137), (20, 1, 500, -100, -36), (65, 1, 300, 5, 5), (40, 3, 257, -127, 128),
    (40, 1, 1000, -300, -43), (40, 1, 1000, -128, 128), (70, 2, 640, 100, 639), (40, 1, 900, -899, 899),
    (97, 1, 513, -223, 224), (600, 1, 130, -7, 8), (600, 1, 130, -20, 20), (600, 2, 131, -40, 50),
    (600, 1, 130, -60, 60)])
def test_lag_windows(oracle, name, n, C, L, lo, hi):
    form, tol = FORMS[name]
    rng = np.random.default_rng(n + L + hi)
    x = rng.standard_normal((n, C, L + 2)).astype(np.float32)
    x = (x[..., 2:] + x[..., 1:-1] + x[..., :-2]) * np.float32(0.5)  # neighbouring lags correlated
    print(f"case lag window {name} n={n} C={C} L={L} [{lo}, {hi}]", flush=True)
    vp, lp, vn, ln = engine.allpairs_host(x, 0, lo, hi, form=form)
    pi, pj = oracle.packed_pairs(n)
    ref = oracle.pairs_f64(x, pi, pj, lo, hi, circular=False)
    assert np.abs(vp - ref["pos"]).max() <= tol and np.abs(vn - ref["neg"]).max() <= tol
    sp = (ref["pos"] > 1e-3) & (ref["gap_pos"] >= 1e-12)
    sn = (ref["neg"] < -1e-3) & (ref["gap_neg"] >= 1e-12)
    assert np.array_equal(lp[sp], ref["lag_pos"][sp]) and np.array_equal(ln[sn], ref["lag_neg"][sn])


@pytest.mark.parametrize("name", ["bf16x3", "fp16", "fft"])
@pytest.mark.parametrize("lo,hi,at,bad", [(-40, 40, 3, np.nan), (-299, 299, 150, np.nan), (5, 200, 290, np.inf),
                                          (-250, -30, 0, -np.inf), (-299, 299, 0, -np.nan)])
def test_nonfinite_rows(oracle, name, lo, hi, at, bad):
    """A NaN or infinite sample in one channel of one event: that event's pairs
    are (0, lag 0), whichever lags reach the sample; the other pairs keep their
    coefficients."""
    form, tol = FORMS.get(name, (engine.FORM_FFT_F32, 1e-5))
    n, C, L, e = 40, 2, 300, 17
    rng = np.random.default_rng(at + abs(hi))
    x = rng.standard_normal((n, C, L)).astype(np.float32)
    pi, pj = oracle.packed_pairs(n)
    ref = oracle.pairs_f64(x, pi, pj, lo, hi, circular=False)
    x[e, 1, at] = bad
    print(f"case nonfinite {name} [{lo}, {hi}] at {at}", flush=True)
    vp, lp, vn, ln = engine.allpairs_host(x, 1024 if name == "fft" else 0, lo, hi, form=form)
    hit = (pi == e) | (pj == e)
    assert not vp[hit].any() and not lp[hit].any() and not vn[hit].any() and not ln[hit].any()
    assert np.abs(vp - ref["pos"])[~hit].max() <= tol and np.abs(vn - ref["neg"])[~hit].max() <= tol


@pytest.mark.parametrize("sign", [1, -1])
def test_lags_beyond_the_record_capacity(sign):
    """More near ties than records (a band of every value): the pairs beyond the
    capacity keep the lag of their FP32 extremum, also where another lag is within
    16 units in the last place.  Single spikes against events with two spikes of
    0.6875 + 3 and + 6 such units: every product is exact."""
    n, L, w = 5800, 64, 30
    rng = np.random.default_rng(5)
    at = rng.integers(20, 45, n)
    x = np.zeros((n, 1, L), np.float32)
    e = np.arange(n)
    one, two = e[::2], e[1::2]
    x[one, 0, at[one]] = 1.0
    a, b = 0.6875 + 3 * 2.0**-24, 0.6875 + 6 * 2.0**-24
    x[two, 0, at[two]] = a
    x[two, 0, at[two] - 1] = b
    x[two, 0, at[two] + 12] = np.sqrt(1.0 - a * a - b * b)
    x[two] *= sign
    print(f"case records beyond the capacity N={n} L={L} +-{w} sign={sign}", flush=True)
    plan = engine.AllPairsPlan(n, 1, L, 0, -w, w, tie_tol=10.0, form=engine.FORM_LAG_BF16X3)
    out = plan.execute(DeviceArray.from_numpy(x))
    synchronize()
    vp, lp, vn, ln = [o.numpy() for o in out]
    stats = plan.stats()
    plan.close()
    assert stats["tie_overflow"] > 10000
    i, j = np.triu_indices(n)
    v, lag = (vp, lp) if sign > 0 else (-vn, ln)
    k = (i % 2 == 0) & (j % 2 == 1)
    assert np.array_equal(lag[k], at[i[k]] - (at[j[k]] - 1)) and np.abs(v[k] - b).max() <= 2e-7
    k = (i % 2 == 1) & (j % 2 == 0)
    assert np.array_equal(lag[k], at[i[k]] - 1 - at[j[k]]) and np.abs(v[k] - b).max() <= 2e-7
    k = (i % 2 == 0) & (j % 2 == 0)
    assert np.array_equal(lp[k], at[i[k]] - at[j[k]]) and (vp[k] == 1.0).all()


@pytest.mark.parametrize("name", ["bf16x3", "fp16"])
@pytest.mark.parametrize("band,block", [(32, 32), (96, 64), (128, 224)])
def test_row_operands_in_bands(name, band, block):
    """Row operands held for some events at a time, as where memory is short: the
    same bits as with all of them, for plans and tiled runs; rows shorter than L,
    demeaned, one of them with a NaN; two executes."""
    n, C, L, in_len, lo, hi = 203, 2, 700, 650, -70, 333
    form, _ = FORMS[name]
    x = np.random.default_rng(band).standard_normal((n, C, in_len)).astype(np.float32) + np.float32(0.5)
    x[70, 1, 5] = np.nan
    print(f"case row bands {name} N={n} C={C} L={L} [{lo}, {hi}] band={band} block={block}", flush=True)
    d = DeviceArray.from_numpy(x)
    plan = engine.AllPairsPlan(n, C, L, 0, lo, hi, demean=True, form=form)
    want = [o.numpy() for o in plan.execute(d)]
    plan.lib.sxc_plan_destroy(plan.handle)
    assert plan.lib.sxc_lag_plan_create_band(ctypes.byref(plan.desc), band, ctypes.byref(plan.handle)) == 0
    for _ in range(2):
        out = plan.execute(d)
        synchronize()
        assert all(np.array_equal(w, o.numpy()) for w, o in zip(want, out))
    plan.close()
    run = tiled.TiledRun(n, C, L, lo, hi, form=form, block=block, demean=True)
    run.lib.sxc_tiled_destroy(run.handle)
    assert run.lib.sxc_tiled_create_band(ctypes.byref(plan.desc), block, 0, band, ctypes.byref(run.handle)) == 0
    coef, lag = np.zeros((n, n), np.float16), np.zeros((n, n), np.int16)
    i, j = np.triu_indices(n)
    for _ in range(2):
        run.start(d)
        tiled.assemble(run, coef, lag)
        assert np.array_equal(coef[i, j], want[0].astype(np.float16)) and np.array_equal(lag[i, j], want[1])
    run.close()


@pytest.mark.parametrize("name,n,C,L,lo,hi", [
    ("bf16x3", 512, 3, 1400, -20, 20), ("bf16x3", 520, 3, 1397, -15, 17), ("bf16x3", 512, 3, 1400, -7, 40),
    ("bf16x3", 512, 1, 4100, 100, 140), ("bf16x3", 512, 3, 1400, -1399, -1360), ("bf16x3", 600, 3, 2500, 60, 95),
    ("bf16x3", 1200, 3, 4096, -31, 31), ("bf16x3", 1200, 3, 4096, -50, 50), ("bf16x3", 1200, 3, 4096, 0, 0),
    ("bf16x3", 1200, 3, 4096, -4095, -4080), ("fp16", 1200, 1, 4096, -3, -3), ("fp16", 1200, 3, 2500, -10, 11),
    ("fp16", 1200, 3, 4096, -23, 20), ("fp16", 1200, 3, 4096, -24, 25)])
def test_few_lags_on_many_samples(oracle, name, n, C, L, lo, hi):
    """Windows that run on the tile kernel (jobs that fill the CUs, one to seven
    blocks of 16 lags from a first lag that is 1 modulo 8 on): a sample of the
    pairs against FP64 direct sums, a row with a NaN, and a tiled run against the
    packed execute."""
    form, tol = FORMS[name]
    rng = np.random.default_rng(n + L + hi)
    x = rng.standard_normal((n, C, L + 2)).astype(np.float32)
    x = (x[..., 2:] + x[..., 1:-1] + x[..., :-2]) * np.float32(0.5)
    bad = x.copy()
    bad[7, 0, L // 2] = np.nan
    print(f"case few lags {name} n={n} C={C} L={L} [{lo}, {hi}]", flush=True)
    plan = engine.AllPairsPlan(n, C, L, 0, lo, hi, form=form)
    d = DeviceArray.from_numpy(bad)
    vp, lp, vn, ln = [o.numpy() for o in plan.execute(d)]
    plan.close()
    pi, pj = oracle.packed_pairs(n)
    hit = (pi == 7) | (pj == 7)
    assert not vp[hit].any() and not lp[hit].any() and not vn[hit].any() and not ln[hit].any()
    k = np.unique(np.concatenate([np.flatnonzero(~hit)[-40:], rng.choice(np.flatnonzero(~hit), 3000)]))
    ref = oracle.pairs_f64(x, pi[k], pj[k], lo, hi, circular=False)
    assert np.abs(vp[k] - ref["pos"]).max() <= tol and np.abs(vn[k] - ref["neg"]).max() <= tol
    sp = (ref["pos"] > 1e-3) & (ref["gap_pos"] >= 1e-12)
    sn = (ref["neg"] < -1e-3) & (ref["gap_neg"] >= 1e-12)
    assert np.array_equal(lp[k][sp], ref["lag_pos"][sp]) and np.array_equal(ln[k][sn], ref["lag_neg"][sn])
    run = tiled.TiledRun(n, C, L, lo, hi, form=form, block=256)
    coef, lag = np.zeros((n, n), np.float16), np.zeros((n, n), np.int16)
    run.start(d)
    tiled.assemble(run, coef, lag)
    run.close()
    assert np.array_equal(coef[pi, pj], vp.astype(np.float16)) and np.array_equal(lag[pi, pj], lp)
