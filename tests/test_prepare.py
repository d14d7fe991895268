"""The bindings' padding against its definition, row by row: each trace (and
its flip) zero-padded to P = 1 << L.bit_length() and cast to float32 through
float, over element types, containers, memory orders and uneven lengths."""
import numpy as np
import pytest

from seismic_amd import correlation_lib


def _row(x, width):
    return np.pad(x, (0, width - x.shape[0]), "constant").astype(float).astype(np.float32)


def _events(kind):
    rng = np.random.default_rng(4)
    x = rng.standard_normal((6, 300)) * 1e4
    ragged = np.empty(4, dtype=object)
    for i, n in enumerate((300, 12, 512, 301)):
        ragged[i] = rng.standard_normal(n).astype(np.float32)
    return {"float64": x, "float32": x.astype(np.float32), "float16": x.astype(np.float16),
            "int64": (x * 1e6).astype(np.int64) + 2**53, "int32": x.astype(np.int32), "bool": x > 0,
            "big endian": x.astype(">f4"), "fortran": np.asfortranarray(x), "strided": x[::2, ::-3], "list": list(x),
            "nan": np.where(x > 0, np.nan, x), "ragged": ragged, "one": x[:1, :1]}[kind]


@pytest.mark.parametrize("kind", ["float64", "float32", "float16", "int64", "int32", "bool", "big endian", "fortran",
                                  "strided", "list", "nan", "ragged", "one"])
def test_prepare_rows(kind):
    ev = _events(kind)
    n, L, P, padded, rev, outs = correlation_lib.prepare(ev)
    rows = [np.asarray(e) for e in ev]
    assert (n, L) == (len(rows), rows[0].shape[0]) and P == 1 << L.bit_length()
    assert padded.dtype == rev.dtype == np.float32 and padded.shape == rev.shape == (n, P)
    for i, r in enumerate(rows):
        assert np.array_equal(padded[i], _row(r, P), equal_nan=True)
        assert np.array_equal(rev[i], _row(np.flip(r, 0), P), equal_nan=True)
    assert all(o.shape == (n * (n + 1) // 2,) for o in outs)


def test_prepare_refuses_rows_longer_than_the_period():
    ev = np.empty(2, dtype=object)
    ev[0], ev[1] = np.zeros(100, np.float32), np.zeros(200, np.float32)  # P = 128
    with pytest.raises(ValueError):
        correlation_lib.prepare(ev)


@pytest.mark.parametrize("shape", [(0, 0), (0, 5), (3, 0)])
def test_prepare_without_events_or_samples(shape):
    """Left to the library, whose message reaches the caller."""
    n, L, P, padded, rev, outs = correlation_lib.prepare(np.zeros(shape, np.float32))
    assert (n, L, P) == (shape[0], 0, 1) and padded.shape == rev.shape == (n, 1)
    assert not padded.any() and not rev.any() and all(o.shape == (n * (n + 1) // 2,) for o in outs)


def test_no_events_reach_the_library():
    with pytest.raises(RuntimeError, match="n_events must be >= 1"):
        correlation_lib.compute_correlation(np.zeros((0, 5), np.float32), 1, 1, 0.0)
