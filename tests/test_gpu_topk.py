"""The server's top-k over catalogs at the edges of its waves (512 columns each,
4096 a turn) and of its column slices (16384 and up): a catalog of a few
distinct events repeated, so that equal values come in every wave and slice,
and must be returned in the order of their columns."""
import numpy as np
import pytest

from seismic_amd import serving

from test_serving import oracle_topk

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n_cat,k,distinct", [(1, 1, 1), (3, 3, 3), (64, 32, 5), (65, 10, 7), (511, 8, 64),
                                              (513, 32, 3), (4096, 10, 4096 // 4), (4097, 16, 600), (32768, 32, 1500),
                                              (40001, 10, 8000)])
def test_topk_order_of_equal_values(n_cat, k, distinct):
    rng = np.random.default_rng(n_cat)
    cycle = rng.standard_normal((distinct, 1, 64)).astype(np.float32)
    cat = cycle[np.arange(n_cat) % distinct]
    print(f"case topk n_cat={n_cat} k={k} distinct={distinct}", flush=True)
    srv = serving.Server(cat, max_query_len=64, top_k=k, max_batch_events=4, n_slots=1)
    q = np.concatenate([cycle[:1], cycle[-1:], np.zeros((1, 1, 64), np.float32)])
    v, _, idx, _ = srv.wait(srv.submit(q, np.array([64, 64, 64], np.int32)))
    srv.close()
    ref = oracle_topk(q[:2], [64] * 2, cycle[:min(distinct, n_cat)], min(distinct, n_cat))
    for e in range(2):
        # the distinct events best first, each with its columns in order, cut at k
        want = [c for t in ref[e] for c in range(t[2], n_cat, distinct)][:k]
        val = [t[0] for t in ref[e] for c in range(t[2], n_cat, distinct)][:k]
        assert np.abs(v[e] - val).max() <= 1e-5
        gaps = np.diff([t[0] for t in ref[e]])
        if len(gaps) == 0 or np.abs(gaps[:k]).min() > 2e-5:  # distinct values told apart in FP32
            assert idx[e].tolist() == want
        same = v[e][1:] == v[e][:-1]
        assert (v[e][1:] <= v[e][:-1]).all() and (idx[e][1:][same] > idx[e][:-1][same]).all()
        assert len(set(idx[e].tolist())) == k
    assert not v[2].any() and idx[2].tolist() == list(range(k))  # a silent query: all 0, by column
