"""Workloads that stand for what programs do with this framework, through its
public entry points: device-resident all-pairs plans (FP32-FFT and MFMA
lag-window forms), the drop-in host call, the serving loop and the tiled
N x N run.

`listed()` gives the named cases, `draw(rng)` more cases of the same ranges;
`prepare(case, seed)` makes what a program holds before the call (events on
the device or on the host, the plan, the server), `run(state)` makes one pass,
`work(case)` says what a pass cannot do without and `exact(case, seed)` gives
the same outputs in 64 bits, without this repository's code.

Events are synthetic in the manner of seismic_amd.synth: white noise
band-passed to 1-20 Hz at 100 Hz plus a 5 Hz Ricker wavelet at a random
offset, demeaned.  torch is imported first, so that the engine binds to the
HIP runtime torch has loaded and both see one device.
"""
import math

import numpy as np
import torch

from seismic_amd import correlation_lib, engine, serving, tiled
from seismic_amd.device import DeviceArray

PERIODS = (1024, 2048, 3072, 4096, 5120, 6144, 8192)
DEV = "cuda"


def listed():
    return [
        # The smallest call: sixteen one-channel events, every lag -- a quick
        # look at one earthquake cluster, where launches and latency count.
        _fft("fft_16_events", 16, 1, 1024, 2048, -1023, 1024),
        # A swarm of a day on a short lag window, three channels, a trace
        # length that is no power of two.
        _fft("fft_200_window", 200, 3, 1000, 2048, -100, 100),
        # The benchmark's workload: 4096 events, three channels, every lag.
        _fft("fft_4096_full", 4096, 3, 2048, 4096, -2047, 2048),
        # A catalog scanned on the benchmark's +-512 window, odd event count.
        _fft("fft_3001_window", 3001, 3, 2048, 4096, -512, 512),
        # Long traces of one channel, every lag, the largest period.
        _fft("fft_1501_long", 1501, 1, 4096, 8192, -4095, 4096),
        # A mixed-radix period with FP64 mean removal, two channels.
        _fft("fft_1111_demean", 1111, 2, 1500, 3072, -1499, 1499, demean=True),
        # The reference's own call on host arrays (padding, copies, compute).
        {"name": "dropin_1024", "kind": "dropin", "n": 1024, "len": 2048, "shift": 2048},
        # The matrix-core forms on the benchmark's window.
        _lag("bf16x3_1500", "bf16x3", 1500, 3, 2048, -512, 512),
        # One channel, long traces, FP16 product, odd event count.
        _lag("fp16_2001_long", "fp16", 2001, 1, 4096, -512, 512),
        # Serving: one new event, and a 64-event request of uneven lengths,
        # against a resident catalog.
        _serve("serve_1", 1, 4096, 3, 2048, 4096),
        _serve("serve_64", 64, 4096, 3, 2048, 4096),
        # The tiled N x N run on the +-1024 window, blocks streamed to the host.
        {"name": "tiled_1000", "kind": "tiled", "n": 1000, "c": 1, "len": 4096, "lo": -1024, "hi": 1024,
         "block": 512, "form": "bf16x3"},
    ]


def _fft(name, n, c, length, period, lo, hi, demean=False):
    return {"name": name, "kind": "fft", "n": n, "c": c, "len": length, "period": period, "lo": lo, "hi": hi,
            "demean": demean}


def _lag(name, form, n, c, length, lo, hi, demean=False):
    return {"name": name, "kind": "lag", "form": form, "n": n, "c": c, "len": length, "lo": lo, "hi": hi,
            "demean": demean}


def _serve(name, n, catalog, c, length, longest):
    return {"name": name, "kind": "serve", "n": n, "catalog": catalog, "c": c, "len": length, "longest": longest}


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case: sizes spread over the ranges above (over their
    logarithm), odd ones among them, within the listed cases' cost."""
    kind = rng.choice(("fft", "fft", "fft", "lag", "lag", "dropin", "serve", "tiled"))
    while True:
        if kind == "fft":
            length = _log(rng, 200, 4096)
            c = rng.randint(1, 4)
            if rng.random() < 0.5:  # the bindings' rule
                period = max(1024, min(8192, 1 << length.bit_length()))
            else:  # the smallest period without wrap-around at any lag
                period = next(p for p in PERIODS if p >= min(8192, 2 * length - 1))
            n = _log(rng, 12, 4096)
            if rng.random() < 0.5:
                lo, hi = max(1 - period // 2, 1 - length), min(period // 2, length)
            else:
                hi = min(_log(rng, 20, 1024), period // 2, length - 1)
                lo = -min(hi, period // 2 - 1) + rng.randint(0, 1)
            case = _fft("", n, c, length, period, lo, hi, demean=rng.random() < 0.25)
        elif kind == "lag":
            length = _log(rng, 200, 4096)
            hi = min(_log(rng, 20, 1024), length - 1)
            case = _lag("", rng.choice(("bf16x3", "fp16")), _log(rng, 40, 2200), rng.randint(1, 3), length,
                        -hi + rng.randint(0, 1), hi, demean=rng.random() < 0.25)
        elif kind == "dropin":
            length = _log(rng, 500, 4000)  # the bindings' periods 1024 .. 4096 (length 512 and up)
            length = max(length, 512)
            shift = length if rng.random() < 0.5 else min(length, _log(rng, 50, 1000))
            shift = min(shift, (1 << length.bit_length()) - length)
            case = {"name": "", "kind": "dropin", "n": _log(rng, 16, 1400), "len": length, "shift": shift}
        elif kind == "serve":
            case = _serve("", _log(rng, 1, 64), _log(rng, 600, 4096), rng.randint(1, 3), _log(rng, 600, 2048),
                          _log(rng, 600, 4096))
        else:
            length = _log(rng, 600, 4096)
            hi = min(_log(rng, 60, 1024), length - 1)
            case = {"name": "", "kind": "tiled", "n": _log(rng, 100, 1000), "c": 1, "len": length, "lo": -hi,
                    "hi": hi, "block": rng.choice((256, 512)), "form": rng.choice(("bf16x3", "fp16"))}
        del case["name"]
        if _fits(case):
            return case


def _fits(case):
    """Within the cost of the listed cases of its kind."""
    limit = max(work(c)["flops"] for c in listed() if c["kind"] == case["kind"])
    return work(case)["flops"] <= limit


# ---------------------------------------------------------------- inputs

def _events(n, c, length, seed):
    """[n, c, length] float32 on the device."""
    g = torch.Generator(device=DEV)
    g.manual_seed(seed)
    fs, f0 = 100.0, 5.0
    freq = torch.fft.rfftfreq(length, d=1.0 / fs, device=DEV)
    gain = torch.clamp((freq - 0.5) / 0.5, 0, 1) * torch.clamp((22.0 - freq) / 2.0, 0, 1)
    half = 40
    off = torch.randint(half, max(half + 1, length - half), (n, 1, 1), generator=g, device=DEV)
    snr = torch.rand((n, c, 1), generator=g, device=DEV) * 9.5 + 0.5
    out = torch.empty((n, c, length), dtype=torch.float32, device=DEV)
    step = max(1, (1 << 24) // (c * length))
    for a in range(0, n, step):
        b = min(n, a + step)
        x = torch.randn((b - a, c, length), generator=g, device=DEV)
        x = torch.fft.irfft(torch.fft.rfft(x) * gain, n=length)
        rms = x.square().mean(-1, keepdim=True).sqrt()
        t = (torch.arange(length, device=DEV) - off[a:b]).to(torch.float32)
        u = (math.pi * f0 / fs * t) ** 2
        w = (1.0 - 2.0 * u) * torch.exp(-u) * (t.abs() <= half)
        x = x + snr[a:b] * rms * w
        out[a:b] = x - x.mean(-1, keepdim=True)
    return out


def _case_events(case, seed):
    """The case's float32 events as they reach the framework."""
    x = _events(case["n"], case.get("c", 1), case["len"], seed)
    if case.get("demean"):  # raw counts with an offset, which the plan removes
        g = torch.Generator(device=DEV)
        g.manual_seed(seed + 7)
        x = x + torch.randn((x.shape[0], x.shape[1], 1), generator=g, device=DEV) * x.std()
    return x


def _queries(case, seed):
    """A request's events (zero beyond each one's length) and lengths."""
    rng = np.random.Generator(np.random.PCG64(seed))
    lens = rng.integers(min(512, case["longest"]), case["longest"] + 1, size=case["n"]).astype(np.int32)
    x = _events(case["n"], case["c"], case["longest"], seed + 1).cpu().numpy()
    for e, m in enumerate(lens):
        x[e, :, m:] = 0.0
    return x, lens


class _Shared:
    """What torch needs to see a DeviceArray without a copy."""

    def __init__(self, a):
        self.owner = a
        self.__cuda_array_interface__ = {"shape": a.shape, "typestr": a.dtype.str, "data": (a.ptr, False),
                                         "version": 2, "strides": None}


def _tensor(a):
    return torch.as_tensor(_Shared(a), device=DEV)


def _device(x):
    return DeviceArray.from_numpy(x.cpu().numpy())


_FORMS = {"bf16x3": engine.FORM_LAG_BF16X3, "fp16": engine.FORM_LAG_FP16}


def prepare(case, seed):
    kind = case["kind"]
    if kind in ("fft", "lag"):
        traces = _device(_case_events(case, seed))
        plan = engine.AllPairsPlan(case["n"], case["c"], case["len"], case.get("period", 0), case["lo"], case["hi"],
                                   demean=case["demean"],
                                   form=engine.FORM_FFT_F32 if kind == "fft" else _FORMS[case["form"]])
        out = plan.alloc_outputs()
        return {"kind": kind, "plan": plan, "traces": traces, "out": out, "seen": [_tensor(a) for a in out]}
    if kind == "dropin":
        return {"kind": kind, "events": _case_events(case, seed)[:, 0].cpu().numpy(), "shift": case["shift"]}
    if kind == "serve":
        catalog = _events(case["catalog"], case["c"], case["len"], seed + 2).cpu().numpy()
        server = serving.Server(catalog, case["longest"], top_k=10, max_batch_events=64, n_slots=2)
        events, lens = _queries(case, seed)
        return {"kind": kind, "server": server, "events": events, "lens": lens}
    run_ = tiled.TiledRun(case["n"], case["c"], case["len"], case["lo"], case["hi"], form=_FORMS[case["form"]],
                          block=case["block"])
    n = case["n"]
    return {"kind": kind, "run": run_, "traces": _device(_case_events(case, seed)),
            "coef": np.empty((n, n), np.float16), "lag": np.empty((n, n), np.int16)}


def run(s):
    kind = s["kind"]
    if kind in ("fft", "lag"):
        s["plan"].execute(s["traces"], out=s["out"])
        return dict(zip(("pos", "lag_pos", "neg", "lag_neg"), s["seen"]))
    if kind == "dropin":
        return dict(zip(("pos", "lag_pos", "neg", "lag_neg"),
                        correlation_lib.compute_correlation(s["events"], s["shift"], 1, 0.0)))
    if kind == "serve":
        values, lags, index, _ = s["server"].wait(s["server"].submit(s["events"], s["lens"]))
        return {"value": values, "lag": lags, "index": index}
    s["run"].start(s["traces"])
    tiled.assemble(s["run"], s["coef"], s["lag"])
    return {"coef": s["coef"], "lag": s["lag"]}


# ---------------------------------------------------------------- work

def _transform(n):
    """Operations of a real transform of n values."""
    return 2.5 * n * math.log2(n)


def work(case):
    kind = case["kind"]
    n, c, length = case["n"], case.get("c", 1), case["len"]
    pairs = n * (n + 1) // 2
    if kind in ("fft", "dropin"):
        if kind == "fft":
            period, reach = case["period"], max(-case["lo"], case["hi"])
        else:
            period, reach = 1 << length.bit_length(), case["shift"]
        m = min(period, length + reach)  # long enough that no lag of the window wraps around
        flops = n * c * _transform(m) + pairs * (8.0 * c * (m // 2 + 1) + _transform(m))
        return {"bytes": 4.0 * n * c * length + 16.0 * pairs, "flops": flops}
    if kind == "serve":
        m = case["longest"] + case["len"]
        flops = n * c * _transform(m) + n * case["catalog"] * (8.0 * c * (m // 2 + 1) + _transform(m))
        return {"bytes": 4.0 * c * (case["catalog"] * length + n * case["longest"]) + 120.0 * n, "flops": flops}
    lags = sum(length - abs(v) for v in range(case["lo"], case["hi"] + 1))
    return {"bytes": 4.0 * n * c * length + (4.0 * n * n if kind == "tiled" else 16.0 * pairs),
            "flops": 2.0 * lags * c * pairs}


# ---------------------------------------------------------------- 64 bits

def _unit(x):
    """Rows in 64 bits over their norms (a silent row stays zero)."""
    x = x.to(torch.float64)
    e = x.square().sum(-1, keepdim=True).sqrt()
    return torch.where(e > 0, x / e, torch.zeros_like(x))


def _extremes(rows, cols, period, lags, first_col):
    """Largest coefficient above 0 and smallest below 0 of every row against
    its columns from first_col(row) on, one after another in two tensors.
    The pairs go through one transform shape in fixed batches."""
    xr, xc = torch.fft.rfft(rows, n=period), torch.fft.rfft(cols, n=period).conj()
    at = torch.arange(lags[0], lags[1] + 1, device=DEV) % period
    first = torch.tensor([first_col(i) for i in range(rows.shape[0])], device=DEV)
    count = cols.shape[0] - first
    i = torch.repeat_interleave(torch.arange(rows.shape[0], device=DEV), count)
    start = torch.cumsum(count, 0) - count
    j = torch.arange(i.shape[0], device=DEV) - start[i] + first[i]
    step = (1 << 26) // period
    pos, neg = torch.empty(i.shape[0], dtype=torch.float64, device=DEV), torch.empty_like(i, dtype=torch.float64)
    y = torch.zeros((step, xr.shape[-1]), dtype=torch.complex128, device=DEV)
    for a in range(0, i.shape[0], step):
        b = min(i.shape[0], a + step)
        y[:b - a] = xr[i[a:b], 0] * xc[j[a:b], 0]
        for c in range(1, rows.shape[1]):
            y[:b - a] += xr[i[a:b], c] * xc[j[a:b], c]
        w = torch.fft.irfft(y, n=period)[:b - a, at] / rows.shape[1]
        pos[a:b] = w.amax(-1).clamp(min=0.0)
        neg[a:b] = w.amin(-1).clamp(max=0.0)
    return pos, neg


def exact(case, seed):
    kind = case["kind"]
    if kind == "serve":
        q, _ = _queries(case, seed)
        cat = _events(case["catalog"], case["c"], case["len"], seed + 2)
        period = 1 << (case["longest"] + case["len"]).bit_length()
        pos, _ = _extremes(_unit(torch.from_numpy(q).to(DEV)), _unit(cat), period,
                           (1 - case["len"], case["longest"] - 1), lambda i: 0)
        top = pos.view(case["n"], case["catalog"]).topk(10).values
        return {"value": top.cpu(), "lag": None, "index": None}
    x = _case_events(case, seed).to(torch.float64)
    if case.get("demean"):
        # the plan subtracts the mean in 64 bits and holds the samples in 32
        x = (x - x.mean(-1, keepdim=True)).to(torch.float32)
    length = case["len"]
    if kind == "fft":
        period, lags = case["period"], (case["lo"], case["hi"])
    elif kind == "dropin":
        period, lags = 1 << length.bit_length(), (1 - case["shift"], case["shift"])
    else:
        period, lags = 2 << length.bit_length(), (case["lo"], case["hi"])
    u = _unit(x)
    pos, neg = _extremes(u, u, period, lags, lambda i: i)
    if kind == "tiled":
        full = torch.zeros((case["n"], case["n"]), dtype=torch.float64, device=DEV)
        r, c = torch.triu_indices(case["n"], case["n"], device=DEV)
        full[r, c] = pos
        full[c, r] = pos
        return {"coef": full.cpu(), "lag": None}
    return {"pos": pos.cpu(), "lag_pos": None, "neg": neg.cpu(), "lag_neg": None}
