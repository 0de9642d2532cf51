"""Host-pointer calls through the cache's pinned scratch, which the kernels read
and write in place: every call of a series on one cache sees its own inputs and
returns its own result, around the 1 MiB up to which an input is read there and
around the scratch's 4 MiB limit (where the buffers are copied instead)."""
import numpy as np
import pytest

import oracle as O
from conftest import tol_close
from test_gpu_headline import E  # noqa: F401

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("d,n_kv,n_q,L", [
    (128, 8, 8, 300), (64, 2, 6, 77), (128, 2, 10, 1000), (64, 32, 32, 257),
    (128, 32, 32, 8190), (64, 4, 32, 8192), (128, 32, 32, 32600), (128, 32, 32, 32800)])
def test_series_of_calls(E, d, n_kv, n_q, L):  # noqa: F811
    rng = np.random.default_rng(0xEA4B + L + d)
    rounds = 2 if L > 10000 else 6
    g, o = E.Cache(1, n_kv, d, L + rounds), O.OracleCache(1, n_kv, d, L + rounds)
    data = rng.standard_normal((2, n_kv, L, d), dtype=np.float32)
    for c in (g, o):
        c.load_raw(data, L)
    for _ in range(rounds):
        new = rng.standard_normal((2, n_kv, 1, d), dtype=np.float32)
        for c in (g, o):
            for kv in (0, 1):
                c.append(new[kv], 0, kv, 1)
            c.advance(1)
        q = rng.standard_normal((n_q, d), dtype=np.float32)
        sg, so = g.attention_scores(q, 0, n_q, n_kv), o.attention_scores(q, 0, n_q, n_kv)
        assert np.array_equal(sg.view(np.uint32), so.view(np.uint32))
        w = O.softmax_rows(so)
        # the bar of the unfused output and of the fused call (conftest)
        for got, want in ((g.attention_output(w, 0, n_q, n_kv), o.attention_output(w, 0, n_q, n_kv)),
                          (g.attention_fused(q, 0, n_q, n_kv), o.attention_fused(q, 0, n_q, n_kv))):
            ok, err, bad = tol_close(got, want)
            assert ok, (err, bad)
    for a, b in zip(g.read_planes(0, 1), o.read_planes(0, 1)):
        assert np.array_equal(a.view(np.uint8), b.view(np.uint8))
    g.free()
    o.free()
