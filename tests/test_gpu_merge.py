"""The chunk merge inside the fused launch and its V-sum form at their edges:
one chunk (written directly), 2, 8 and 9 (both batch sizes), 16, one and two
outputs per thread, more one-chunk units than counters, and empty sequences.
Both entry points give the same bits; results meet the reference bar."""
import numpy as np
import pytest

import oracle as O
from conftest import tol_close
from test_gpu_headline import (E, batch_call, build_batch, chan_k,  # noqa: F401
                               compare_sequences, n_cu, say)

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("n_kv,n_q,n_seq,L,chunks", [
    (8, 8, 1, 100, 1), (8, 32, 1, 128, 1), (4, 8, 1, 200, 2), (8, 32, 1, 1024, 8),
    (8, 8, 1, 1025, 9), (8, 32, 1, 1025, 9), (4, 16, 1, 2048, 16), (32, 32, 16, 300, 1),
    (32, 32, 9, 3071, 1), (32, 32, 9, 3072, 2)])
def test_merge_edges(E, d, n_kv, n_q, n_seq, L, chunks):  # noqa: F811
    gs, os_ = build_batch(E, 0xEA4B + 800 + d + L, n_seq, n_kv, d, [L] * n_seq, L + 3, chan_k)
    plan = E.fused_plan(gs, n_q, n_kv)
    say("merge: plan", plan)
    if n_cu() == 256:
        assert plan["chunks"] == chunks
    rng = np.random.default_rng(0xEA4B + 801 + d)
    q = rng.standard_normal((n_seq, n_q, d), dtype=np.float32)
    out = batch_call(E, "eakv_attention_fused_batch_device", gs, q, n_q, n_kv)
    out_na = batch_call(E, "eakv_attention_fused_batch_device_noalloc", gs, q, n_q, n_kv)
    assert np.array_equal(out.view(np.uint32), out_na.view(np.uint32))
    compare_sequences(os_, q, out, n_q, n_kv, [L] * n_seq)
    w = O.softmax_rows(os_[0].attention_scores(q[0], 0, n_q, n_kv))
    w[0, 0] = -w[0, 0]
    ok, err, bad = tol_close(gs[0].attention_output(w, 0, n_q, n_kv),
                             os_[0].attention_output(w, 0, n_q, n_kv))
    assert ok, (err, bad)
    w[n_q - 1, 0] = np.inf
    got = gs[0].attention_output(w, 0, n_q, n_kv)
    assert not np.isfinite(got[n_q - 1]).any() and np.isfinite(got[:n_q - 1]).all()
    for g in gs:
        g.free()


def test_empty_batch(E):  # noqa: F811
    gs = [E.Cache(1, 2, 64, 40) for _ in range(3)]
    q = np.ones((3, 4, 64), np.float32)
    for fn in ("eakv_attention_fused_batch_device", "eakv_attention_fused_batch_device_noalloc"):
        assert np.isnan(batch_call(E, fn, gs, q, 4, 2)).all()
    for g in gs:
        g.free()


@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("n_kv,n_q,L,chunks", [
    (8, 8, 100, 1), (8, 32, 100, 1), (8, 8, 640, 5), (8, 32, 640, 5), (8, 32, 1024, 8),
    (8, 64, 1024, 8), (8, 8, 1500, 12), (4, 16, 2048, 16), (2, 8, 9000, 36)])
def test_infinite_partials(E, d, n_kv, n_q, L, chunks):  # noqa: F811
    """One group of V near the largest float in every token, with equal
    scores: its sums overflow in every chunk, and both entry points return the
    reference's infinity (a sum padded with infinity times 0 would be NaN)."""
    rng = np.random.default_rng(0xEA4B + 820 + L)
    data = rng.standard_normal((1, 2, n_kv, L, d), dtype=np.float32)
    data[0, 1, 1, :, :64] = np.float32(2e38)
    g, o = E.Cache(1, n_kv, d, L + 4), O.OracleCache(1, n_kv, d, L + 4)
    for c in (g, o):
        c.load_raw(data, L)
    plan = E.fused_plan([g], n_q, n_kv)
    say("infinite partials: plan", plan)
    if n_cu() == 256:
        assert plan["chunks"] == chunks
    q = np.zeros((1, n_q, d), np.float32)
    ref = o.attention_fused(q[0], 0, n_q, n_kv)
    inf = np.isinf(ref)
    assert inf.any() and np.isfinite(ref[~inf]).all()
    outs = [batch_call(E, "eakv_attention_fused_batch_device" + s, [g], q, n_q, n_kv)[0]
            for s in ("", "_noalloc")]
    for out in outs:
        assert np.array_equal(out[inf], ref[inf])
        ok, err, bad = tol_close(out[~inf], ref[~inf])
        assert ok, (err, bad)
    assert np.array_equal(outs[0].view(np.uint32), outs[1].view(np.uint32))
    g.free()
    o.free()


@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("n_q,L", [(8, 100), (32, 100), (64, 100), (32, 1024), (64, 1500),
                                   (32, 4096)])
def test_buffers_aligned_to_4_bytes(E, d, n_q, L):  # noqa: F811
    """Queries, weights, outputs and scores at addresses that are only 4-byte
    aligned, one chunk (stored from the chunk itself) and several: the same bits
    as at aligned addresses, and nothing beside the results touched."""
    from eakv_amd.hipmem import DeviceArray
    n_kv = 8
    rng = np.random.default_rng(0xEA4B + 830 + L + n_q)
    g = E.Cache(1, n_kv, d, L + 4)
    g.load_raw(rng.standard_normal((1, 2, n_kv, L, d), dtype=np.float32), L)
    q = rng.standard_normal((n_q, d), dtype=np.float32)
    w = rng.random((n_q, L), dtype=np.float32)
    one = np.zeros(1, np.float32)
    dq = DeviceArray.from_host(np.concatenate([one, q.ravel()]))
    dq0 = DeviceArray.from_host(q)
    dw = DeviceArray.from_host(np.concatenate([one, w.ravel()]))
    dw0 = DeviceArray.from_host(w)
    lib, hs = E.lib(), E.handles([g])
    q_at, w_at = (dq0.ptr, dq.ptr + 4), (dw0.ptr, dw.ptr + 4)
    calls = [
        (n_q * d, lambda i, p: lib.eakv_attention_fused_batch_device(
            hs, 1, 0, q_at[i], n_q, n_kv, p, None)),
        (n_q * d, lambda i, p: lib.eakv_attention_fused_batch_device_noalloc(
            hs, 1, 0, q_at[i], n_q, n_kv, p, None)),
        (n_q * d, lambda i, p: lib.eakv_attention_output_device(
            g.h, w_at[i], 0, n_q, n_kv, p, None)),
        (n_q * L, lambda i, p: lib.eakv_attention_scores_device(
            g.h, q_at[i], 0, n_q, n_kv, p, None)),
    ]
    for n, call in calls:
        outs = []
        for off in (0, 1):
            buf = DeviceArray.from_host(np.full(n + 2, 7.0, np.float32))
            assert call(off, buf.ptr + 4 * off) == 0, E.last_error()
            g.sync()
            got = buf.download()
            assert got[n + off] == 7.0 and (off == 0 or got[0] == 7.0)
            outs.append(got[off:n + off].view(np.uint32))
        assert np.array_equal(*outs)
    g.free()
