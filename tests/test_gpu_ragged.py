"""Batches of several context lengths on the fused call's proportional chunks.

A batch whose contexts differ enough gives each sequence chunks in proportion
to its length (ragged_kernel, hip/fused.hip) instead of as many chunks for all.
Each case names its chunks of the longest context on 256 CUs and covers an edge:
contexts of one token, around a tile (32) and a round of a block (128), an
empty sequence, more than 16 chunks of a unit or more units than counters (the
merge launch), more blocks than the chip holds at once, one and two quads, both
head_dims, groups split into virtual kv heads.  Outputs are held to the reference bar
(fused_attention.ea:190-373), both entry points to the same bits.
"""
import numpy as np
import pytest

import oracle as O
from conftest import tol_close
from test_gpu_headline import (E, batch_call, build_batch, chan_k,  # noqa: F401
                               compare_sequences, n_cu, say)

pytestmark = pytest.mark.gpu

CASES = [
    (128, 8, 32, [9001, 1, 31, 32, 33, 127, 128, 129, 4000], 15),
    (64, 8, 32, [50000, 1, 500], 56),
    (128, 8, 8, [7000] + [200] * 20, 14),
    (128, 8, 64, [12000] + [300 + i for i in range(29)], 12),
    (128, 8, 40, [30000, 100], 15),
    (64, 4, 32, [30000, 257, 1, 3000, 33], None),
    (128, 2, 64, [10000, 64, 65], 14),
    # 744 one-quad blocks for 512 slots (24 contexts of 192-12289 tokens)
    (128, 8, 32, [int(12289 * 64 ** (-i / 23)) for i in range(24)], 14),
    # more units than counters: the merge launch also from the workspace form
    (64, 12, 12, [2743] + [700] * 24, 4),
]


@pytest.mark.parametrize("d,n_kv,n_q,lens,chunks", CASES)
def test_ragged_batch(E, d, n_kv, n_q, lens, chunks):  # noqa: F811
    say("ragged: build", d, n_q, n_kv, lens)
    gs, os_ = build_batch(E, 0xEA4B + 700 + d + len(lens), len(lens), n_kv, d, lens,
                          max(lens) + 3, chan_k)
    empty = E.Cache(1, n_kv, d, max(lens) + 3)
    n = len(gs) + 1
    batch = gs[:1] + [empty] + gs[1:]
    plan = E.fused_plan(batch, n_q, n_kv)
    say("ragged: plan", plan)
    if n_cu() == 256:
        assert plan["mfma"] == 1 and chunks in (None, plan["chunks"])
        units = n * n_kv * plan["split"]
        assert plan["merge_levels"] == (1 if plan["chunks"] <= 16 and units <= 256 else 0)
    rng = np.random.default_rng(0xEA4B + 701 + d)
    q = rng.standard_normal((n, n_q, d), dtype=np.float32)
    out = batch_call(E, "eakv_attention_fused_batch_device", batch, q, n_q, n_kv)
    out_na = batch_call(E, "eakv_attention_fused_batch_device_noalloc", batch, q, n_q, n_kv)
    again = batch_call(E, "eakv_attention_fused_batch_device", batch, q, n_q, n_kv)
    keep = [0] + list(range(2, n))
    assert np.array_equal(out[keep].view(np.uint32), out_na[keep].view(np.uint32))
    assert np.array_equal(out[keep].view(np.uint32), again[keep].view(np.uint32))
    assert all(np.isnan(x[1]).all() for x in (out, out_na, again))
    compare_sequences(os_, q[keep], out[keep], n_q, n_kv, lens)
    for g in batch:
        g.free()


@pytest.mark.parametrize("d,n_kv,n_q", [(128, 8, 32), (128, 8, 64), (64, 8, 8), (64, 4, 32)])
def test_ragged_nonfinite(E, d, n_kv, n_q):  # noqa: F811
    """A long sequence with a group of V near the largest float (its sums
    overflow: infinity, as the reference), one with a NaN in K (its kv head's
    outputs), and plain ones, which the others leave alone."""
    lens = [9001, 300, 5000, 129]
    rng = np.random.default_rng(0xEA4B + 720 + d + n_q)
    gs, os_ = [], []
    for i, L in enumerate(lens):
        data = rng.standard_normal((1, 2, n_kv, L, d), dtype=np.float32)
        if i == 0:
            data[0, 1, 1, :, :64] = np.float32(2e38)
        if i == 2:
            data[0, 0, 2, L // 2, 0] = np.nan
        gs.append(E.Cache(1, n_kv, d, max(lens)))
        os_.append(O.OracleCache(1, n_kv, d, max(lens)))
        for c in (gs[i], os_[i]):
            c.load_raw(data, L)
    say("ragged non-finite: plan", E.fused_plan(gs, n_q, n_kv))
    q = rng.standard_normal((4, n_q, d), dtype=np.float32)
    q[0] = 0
    out = batch_call(E, "eakv_attention_fused_batch_device", gs, q, n_q, n_kv)
    out_na = batch_call(E, "eakv_attention_fused_batch_device_noalloc", gs, q, n_q, n_kv)
    for i, o in enumerate(os_):
        ref = o.attention_fused(q[i], 0, n_q, n_kv)
        fin = np.isfinite(ref)
        assert fin.all() == (i in (1, 3)) and np.isinf(ref).any() == (i == 0)
        for x in (out[i], out_na[i]):
            assert np.array_equal(np.isnan(x), np.isnan(ref))
            assert np.array_equal(x[np.isinf(ref)], ref[np.isinf(ref)])
            ok, err, bad = tol_close(x[fin], ref[fin])
            assert ok, (i, err, bad)
        assert np.array_equal(out[i][fin].view(np.uint32), out_na[i][fin].view(np.uint32))
    for g in gs:
        g.free()


# The deals at the edges of ragged_chunks' rule where the even deal is one
# chunk each: (d, n_kv, n_q, lens, most chunks of a sequence on 256 CUs)
DEALS = [
    (64, 12, 12, [1241 - 32 * i for i in range(24)], 1),     # a merge launch for 5 rounds
    (64, 12, 12, [2743] + [700] * 24, 4),                    # and for 16
    (128, 8, 64, [7706 - 160 * i for i in range(31)], 1),    # blocks past the slots
    (128, 8, 64, [14435] + [2000] * 17, 8),
    (128, 8, 128, [3661 - 120 * i for i in range(22)], 1),   # units past the slots, short
    (128, 8, 128, [8279 - 300 * i for i in range(18)], 2),   # and long
]


@pytest.mark.parametrize("d,n_kv,n_q,lens,chunks", DEALS)
def test_deal(E, d, n_kv, n_q, lens, chunks):  # noqa: F811
    gs = []
    for L in lens:
        gs.append(E.Cache(1, n_kv, d, max(lens)))
        gs[-1].advance(L)
    plan = E.fused_plan(gs, n_q, n_kv)
    say("deal: plan", plan)
    if n_cu() == 256:
        assert plan["chunks"] == chunks
    for g in gs:
        g.free()
