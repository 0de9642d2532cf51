"""The K-score of groups of q heads (k_score_mfma_kernel, hip/kscore.hip), whose
dots run on the matrix cores, bit for bit against the oracle: group sizes around
its quads of heads, contexts around its 256-token slices and long enough for
two quads a wave (every slice of every quad more than three blocks per CU; at
20000 tokens a block takes several slices, with 10 heads a group the last block's
second quad is empty), and values with denormal products."""
import numpy as np
import pytest

import oracle as O
from test_gpu_headline import E, chan_k  # noqa: F401

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("n_kv,qpk,L,tiny", [
    (2, 2, 1, False), (1, 3, 255, False), (3, 4, 256, False), (2, 5, 257, False),
    (1, 8, 1000, True), (2, 9, 513, False), (1, 17, 300, False),
    (8, 8, 49 * 256 + 1, False), (16, 6, 25 * 256 - 1, False), (8, 4, 27000, False),
    (8, 8, 20000, False), (4, 10, 20000, False)])
def test_group_scores_bit_exact(E, d, n_kv, qpk, L, tiny):  # noqa: F811
    rng = np.random.default_rng(0xEA4B + 31 * qpk + L + d)
    data = np.stack([chan_k(rng, n_kv, L, d), rng.standard_normal((n_kv, L, d), dtype=np.float32)])
    q = rng.standard_normal((n_kv * qpk, d), dtype=np.float32)
    if tiny:
        data *= np.float32(1e-21)
        q *= np.float32(1e-21)
    g, o = E.Cache(1, n_kv, d, L + 5), O.OracleCache(1, n_kv, d, L + 5)
    for c in (g, o):
        c.load_raw(data, L)
    sg = g.attention_scores(q, 0, n_kv * qpk, n_kv)
    so = o.attention_scores(q, 0, n_kv * qpk, n_kv)
    assert np.array_equal(sg.view(np.uint32), so.view(np.uint32)), float(np.abs(sg - so).max())
    if tiny:
        a = np.abs(sg[sg != 0])
        assert a.size and a.min() < 1.1754944e-38
    g.free()
    o.free()
