"""The work that programs have this library do, as cases that can be timed.

Six kinds of work, each through the entry points that a program calls:

  decode   one decode step of a batch of sequences: the step's K and V of all
           layers appended (eakv_append_batch_device), then the fused
           attention of every layer (eakv_attention_fused_batch_device);
           afterwards the contexts are restored, so that a pass can be
           repeated.
  unfused  eakv_attention_scores_device and eakv_attention_output_device of
           every layer.  The row softmax between them is the caller's own
           code; its weights are inputs here.
  host     one layer's step of a program written for the reference's C API:
           eakv_cache_append of K and V, scores and output, all on host
           buffers.
  load     a prompt into an empty cache (eakv_cache_load_raw_device), then its
           planes read back as f32 (eakv_dequantize_range_device), as the
           prompt's own attention takes them.
  extend   the same for a further piece of a prompt, appended layer by layer
           (eakv_cache_append_device) behind what the cache holds.
  ggml     the ggml block type: a matrix quantized row by row, dequantized,
           and multiplied with one vector.

The device-pointer calls run on the library's shared stream (a NULL stream).
"""
import math
import random

import numpy as np
import torch

import eakv_amd

# q heads, kv heads, head_dim
HEADS = [(8, 8, 128), (32, 4, 64), (32, 32, 128), (32, 8, 128), (64, 8, 128), (40, 8, 128),
         (16, 8, 128), (12, 12, 64)]

# Algorithmic bytes of the largest listed case, which no drawn case exceeds
MOST_BYTES = 1.35e9


def listed():
    def decode(name, heads, seqs, ctx, spread, layers):
        return dict(name=name, kind="decode", n_q=heads[0], n_kv=heads[1], d=heads[2], seqs=seqs,
                    ctx=ctx, spread=spread, layers=layers)

    def unfused(name, heads, ctx, layers):
        return dict(name=name, kind="unfused", n_q=heads[0], n_kv=heads[1], d=heads[2], ctx=ctx,
                    layers=layers)

    return [
        # one chat at a short context on a small multi-head model: latency
        # and launches
        decode("decode 8q8kv 2K", (8, 8, 128), 1, 2048, 1, 2),
        # the same on a TinyLlama-shaped model
        decode("decode 32q4kv d64 4K", (32, 4, 64), 1, 4096, 1, 4),
        # a Llama-2-7B-shaped model (one q head per kv head)
        decode("decode 32q32kv 8K", (32, 32, 128), 1, 8192, 1, 4),
        # serving: sequences of one batch have contexts of their own, from a
        # few tokens to the longest
        decode("decode 32q8kv ragged x24", (32, 8, 128), 24, 12289, 64, 4),
        # serving at long contexts of one length
        decode("decode 32q8kv 32K x8", (32, 8, 128), 8, 32768, 1, 4),
        # one long document on a 70B-shaped model
        decode("decode 64q8kv 128K", (64, 8, 128), 1, 131073, 1, 8),
        # programs with a softmax of their own between scores and output
        unfused("unfused 8q8kv 2K", (8, 8, 128), 2048, 1),
        unfused("unfused 32q32kv 8K", (32, 32, 128), 8192, 4),
        unfused("unfused 32q8kv 30K", (32, 8, 128), 30011, 4),
        # the drop-in C API on host buffers
        dict(name="host 8q8kv 2K", kind="host", n_q=8, n_kv=8, d=128, ctx=2048),
        # a prompt's keys and values taken in
        dict(name="load 8kv 8K", kind="load", n_kv=8, d=128, tokens=8192, start=0, layers=4),
        # a weight matrix in the ggml block type
        dict(name="ggml 8192x4096", kind="ggml", rows=8192, cols=4096),
    ]


def _log(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["decode"] * 5 + ["unfused"] * 3 + ["host", "load", "extend", "ggml"])
    if kind == "ggml":
        case = dict(kind=kind, rows=_log(rng, 1, 32768), cols=64 * _log(rng, 1, 256))
        size = "rows"
    else:
        n_q, n_kv, d = rng.choice(HEADS)
        case = dict(kind=kind, n_kv=n_kv, d=d)
        if kind in ("load", "extend"):
            case.update(tokens=_log(rng, 16, 32768), layers=rng.randint(1, 4),
                        start=_log(rng, 1, 8192) if kind == "extend" else 0)
            size = "tokens"
        else:
            case.update(n_q=n_q, ctx=_log(rng, 64, 16384 if kind == "host" else 131072))
            size = "ctx"
            if kind == "decode":
                case.update(seqs=_log(rng, 1, 32), spread=rng.choice([1, 1, 4, 64]))
            if kind != "host":
                case.update(layers=rng.randint(1, 4))
    while work(case)["bytes"] > MOST_BYTES:
        case[size] = case[size] * 2 // 3 + 1
    return case


# ---------------------------------------------------------------- the inputs

def _lengths(case):
    """Contexts of a decode step's sequences, the new token included:
    log-uniform from ctx/spread to ctx, one of them ctx."""
    n, ctx, lo = case["seqs"], case["ctx"], max(1.0, case["ctx"] / case["spread"])
    r = random.Random(n * 1000003 + ctx)
    rest = [max(1, min(ctx, int(round(math.exp(r.uniform(math.log(lo), math.log(ctx)))))))
            for _ in range(n - 1)]
    rest.insert(n // 3, ctx)
    return rest


def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _kv(g, layers, n_kv, tokens, d, chan):
    """K and V f32[layers][2][n_kv][tokens][d]: K with the per-channel scales
    and outlier channels that key caches have, V normal."""
    x = torch.randn(layers, 2, n_kv, tokens, d, generator=g, device="cuda")
    x[:, 0] *= chan
    return x


def _channels(g, n_kv, d):
    """Key channel scales f32[n_kv][1][d]: log-uniform in [0.5, 4], two
    channels of each head ten times larger."""
    c = torch.exp(torch.rand(n_kv, 1, d, generator=g, device="cuda") * math.log(8.0) + math.log(0.5))
    for h in range(n_kv):
        c[h, 0, torch.randperm(d, generator=g, device="cuda")[:2]] *= 10
    return c


def _chunks(case, seed):
    """The cache contents of each sequence in turn (f32 on the device) and the
    generator that the remaining inputs come from."""
    g = _gen(seed)
    chan = _channels(g, case["n_kv"], case["d"])
    if case["kind"] == "decode":
        have = [n - 1 for n in _lengths(case)]
    else:
        have = [case["ctx"] - (case["kind"] == "host")]
    layers = case.get("layers", 1)
    for n in have:
        yield _kv(g, layers, case["n_kv"], n, case["d"], chan), g, chan


def _rest(case, g, chan):
    """The remaining inputs, after the contents: new tokens, queries, weights."""
    layers, n_kv, n_q, d = case.get("layers", 1), case["n_kv"], case["n_q"], case["d"]
    if case["kind"] == "decode":
        n = case["seqs"]
        new = torch.stack([_kv(g, layers, n_kv, 1, d, chan) for _ in range(n)])
        return new, torch.randn(layers, n, n_q, d, generator=g, device="cuda"), None
    new = _kv(g, 1, n_kv, 1, d, chan)[0] if case["kind"] == "host" else None
    q = torch.randn(layers, n_q, d, generator=g, device="cuda")
    # softmax rows of scores with the spread that the keys above give
    w = torch.softmax(3.4 * torch.randn(layers, n_q, case["ctx"], generator=g, device="cuda"), -1)
    return new, q, w


def _must(rc):
    if rc != eakv_amd.EAKV_OK:
        raise RuntimeError("%d: %s" % (rc, eakv_amd.last_error()[1]))


def prepare(case, seed):
    kind = case["kind"]
    L = eakv_amd.lib()
    if kind == "ggml":
        rows, cols = case["rows"], case["cols"]
        g = _gen(seed)
        return dict(case=case, x=torch.randn(rows, cols, generator=g, device="cuda"),
                    y=torch.randn(cols, generator=g, device="cuda"),
                    blocks=torch.empty(rows, cols // 64 * 40, dtype=torch.uint8, device="cuda"),
                    deq=torch.empty(rows, cols, device="cuda"),
                    dot=torch.empty(rows, device="cuda"))
    layers, n_kv, d = case.get("layers", 1), case["n_kv"], case["d"]
    if kind in ("load", "extend"):
        tokens, start = case["tokens"], case["start"]
        g = _gen(seed)
        chan = _channels(g, n_kv, d)
        cache = eakv_amd.Cache(layers, n_kv, d, start + tokens)
        if start:
            old = _kv(g, layers, n_kv, start, d, chan)
            torch.cuda.synchronize()
            _must(L.eakv_cache_load_raw_device(cache.h, old.data_ptr(), start, None))
            cache.sync()
        return dict(case=case, cache=cache, x=_kv(g, layers, n_kv, tokens, d, chan),
                    deq=torch.empty(layers, 2, n_kv, start + tokens, d, device="cuda"))
    caches = []
    for x, g, chan in _chunks(case, seed):
        c = eakv_amd.Cache(layers, n_kv, d, case["ctx"])
        if x.shape[3]:
            torch.cuda.synchronize()
            _must(L.eakv_cache_load_raw_device(c.h, x.data_ptr(), x.shape[3], None))
            c.sync()
        caches.append(c)
        del x
    new, q, w = _rest(case, g, chan)
    st = dict(case=case, caches=caches, new=new, q=q, w=w)
    if kind == "decode":
        st.update(handles=eakv_amd.handles(caches), out=torch.empty_like(q))
    elif kind == "unfused":
        st.update(scores=torch.empty_like(w), out=torch.empty_like(q))
    else:
        st.update(new=new.cpu().numpy(), q=q[0].cpu().numpy(), w=w[0].cpu().numpy(),
                  scores=np.zeros((case["n_q"], case["ctx"]), np.float32),
                  out=np.zeros((case["n_q"], d), np.float32))
    return st


# ------------------------------------------------------------------ one pass

def _decode(st, L, case):
    caches, handles, n = st["caches"], st["handles"], case["seqs"]
    _must(L.eakv_append_batch_device(handles, n, st["new"].data_ptr(), 1, None))
    for c in caches:
        c.advance(1)
    q, out = st["q"].data_ptr(), st["out"].data_ptr()
    step = n * case["n_q"] * case["d"] * 4
    for layer in range(case["layers"]):
        _must(L.eakv_attention_fused_batch_device(handles, n, layer, q + layer * step, case["n_q"],
                                                  case["n_kv"], out + layer * step, None))
    for c in caches:
        c.restore(c.checkpoint() - 1)
    return st["out"]


def _unfused(st, L, case):
    h, n_q, n_kv = st["caches"][0].h, case["n_q"], case["n_kv"]
    q, w, s, o = (st[k].data_ptr() for k in ("q", "w", "scores", "out"))
    row, vec = n_q * case["ctx"] * 4, n_q * case["d"] * 4
    for i in range(case["layers"]):
        _must(L.eakv_attention_scores_device(h, q + i * vec, i, n_q, n_kv, s + i * row, None))
        _must(L.eakv_attention_output_device(h, w + i * row, i, n_q, n_kv, o + i * vec, None))
    return st["scores"], st["out"]


def _host(st, L, case):
    c, n_q, n_kv = st["caches"][0], case["n_q"], case["n_kv"]
    for kv in (0, 1):
        _must(L.eakv_cache_append(c.h, st["new"][kv].ctypes.data, 0, kv, 1))
    c.advance(1)
    L.eakv_attention_scores(c.h, st["q"].ctypes.data, 0, n_q, n_kv, st["scores"].ctypes.data)
    L.eakv_attention_output(c.h, st["w"].ctypes.data, 0, n_q, n_kv, st["out"].ctypes.data)
    c.restore(c.checkpoint() - 1)
    return st["scores"], st["out"]


def _prompt(st, L, case):
    h, x, layers, tokens, start = (st["cache"].h, st["x"], case["layers"], case["tokens"],
                                   case["start"])
    if case["kind"] == "load":
        _must(L.eakv_cache_load_raw_device(h, x.data_ptr(), tokens, None))
    groups = case["n_kv"] * (start + tokens) * case["d"] // 64
    src, dst = x.data_ptr(), st["deq"].data_ptr()
    for i in range(2 * layers):
        if case["kind"] == "extend":
            _must(L.eakv_cache_append_device(h, src + i * case["n_kv"] * tokens * case["d"] * 4,
                                             i // 2, i % 2, tokens, None))
        _must(L.eakv_dequantize_range_device(h, i // 2, i % 2, 0, groups, dst + i * groups * 256,
                                             None))
    return st["deq"]


def _ggml(st, L, case):
    rows, cols = case["rows"], case["cols"]
    x, y, b, q, s = (st[k].data_ptr() for k in ("x", "y", "blocks", "deq", "dot"))
    _must(L.eakv_ggml_quantize_row_device(x, b, rows * cols, None))
    _must(L.eakv_ggml_dequantize_row_device(b, q, rows * cols, None))
    _must(L.eakv_ggml_vec_dot_device(cols, s, 4, b, cols // 64 * 40, y, 0, rows, None))
    return st["blocks"], st["deq"], st["dot"]


_RUN = dict(decode=_decode, unfused=_unfused, host=_host, load=_prompt, extend=_prompt, ggml=_ggml)


def run(state):
    case = state["case"]
    return _RUN[case["kind"]](state, eakv_amd.lib(), case)


# ------------------------------------------------------- what a pass stands for

def work(case):
    """Each input read once, each output written once; a cached token of one
    kv head is 40 bytes for each 64 dims of K and the same of V."""
    kind = case["kind"]
    if kind == "ggml":
        n = case["rows"] * case["cols"]
        # quantize 4 + 40/64 bytes a value, dequantize the same, product 40/64
        return dict(bytes=n * (4 + 0.625) * 2 + n * 0.625 + 4 * (case["rows"] + case["cols"]),
                    flops=12.0 * n)
    layers, n_kv, d = case.get("layers", 1), case["n_kv"], case["d"]
    per = n_kv * d // 64 * 40                           # a token's K (or V) of one layer
    if kind in ("load", "extend"):
        n = case["tokens"]
        seen = case["start"] + n
        return dict(bytes=2.0 * layers * (n * n_kv * d * 4 + n * per + seen * per + seen * n_kv * d * 4),
                    flops=2.0 * layers * n_kv * d * (8 * n + 2 * seen))
    n_q = case["n_q"]
    if kind == "decode":
        seen, n = sum(_lengths(case)), case["seqs"]
        return dict(bytes=float(layers) * (2 * seen * per + n * (2 * n_q * d * 4 + 2 * (n_kv * d * 4 + per))),
                    flops=4.0 * layers * n_q * d * seen)
    seen = case["ctx"]
    # K and V, the scores written, the weights read, queries and output
    b = 2 * seen * per + 2 * n_q * seen * 4 + 2 * n_q * d * 4
    if kind == "host":
        b += 2 * (n_kv * d * 4 + per)
    return dict(bytes=float(layers) * b, flops=4.0 * layers * n_q * d * seen)


def tolerance(case):
    # The quantizer, the dequantizer and the ggml rows are bit-exact by
    # contract: each rounding is fixed by the reference's format and kernels.
    if case["kind"] in ("load", "extend", "ggml"):
        return "exact"
    # f32 softmax and sums over up to 131072 tokens in an order that the
    # implementation chooses: against 64 bits the fused attention is 0.5 to
    # 1.2e-6 off (its exponentials among it), scores and the weighted sum of
    # given weights 0.8 to 2.7e-7 (the 32-bit dequantized values' own rounding
    # is 6e-8).
    return {"rel": 1e-5 if case["kind"] == "decode" else 2e-6}


# ------------------------------------------------------------- in 64 bits

def _quantized(x):
    """The values that the Q4_1 form of x holds, in f64: groups of 64, bias
    the minimum, scale range/15, the nibble's steps each rounded to f32."""
    g = x.reshape(-1, 64)
    mn, mx = g.amin(1, keepdim=True), g.amax(1, keepdim=True)
    r = mx - mn
    pos = r > 0
    # f32 quotients by way of f64 (53 bits are enough for a single rounding)
    scale = torch.where(pos, (r.double() / 15.0).float(), torch.ones_like(r))
    inv = torch.where(pos, (15.0 / r.double()).float(), torch.zeros_like(r))
    n = (g - mn).mul_(inv).add_(0.5).floor_().clamp_(0, 15)
    return (n.double() * scale.double() + mn.double()).reshape(x.shape)


def _attend(k, v, q):
    """softmax(q.k/sqrt(d)).v of f64 k, v [n_kv][t][d] and q [n_q][d], and the scores."""
    n_kv, t, d = k.shape
    s = torch.bmm(q.double().reshape(n_kv, -1, d), k.transpose(1, 2).contiguous()) / math.sqrt(d)
    s = s.reshape(-1, t)
    return s, (None if v is None else _weigh(torch.softmax(s, -1), v))


def _weigh(w, v):
    n_kv, t, d = v.shape
    return torch.bmm(w.double().reshape(n_kv, -1, t), v).reshape(-1, d)


def exact(case, seed):
    kind = case["kind"]
    if kind == "ggml":
        g = _gen(seed)
        x = _quantized(torch.randn(case["rows"], case["cols"], generator=g, device="cuda"))
        y = torch.randn(case["cols"], generator=g, device="cuda")
        return None, x, torch.mv(x, y.double())
    if kind in ("load", "extend"):
        g = _gen(seed)
        layers, n_kv, d = case["layers"], case["n_kv"], case["d"]
        chan = _channels(g, n_kv, d)
        parts = [_kv(g, layers, n_kv, n, d, chan) for n in (case["start"], case["tokens"]) if n]
        return _quantized(torch.cat(parts, 3))
    # contents first (kept as f32), as the inputs after them come last from the generator
    xs = []
    for x, g, chan in _chunks(case, seed):
        xs.append(x)
    new, q, w = _rest(case, g, chan)
    if kind == "unfused":
        got = []
        for i in range(case["layers"]):
            kv = [_quantized(xs[0][i, j]) for j in (0, 1)]
            got.append((_attend(kv[0], None, q[i])[0], _weigh(w[i], kv[1])))
        return torch.stack([a for a, _ in got]), torch.stack([b for _, b in got])
    if kind == "host":
        kv = [_quantized(torch.cat([xs[0][0, j], new[j]], 1)) for j in (0, 1)]
        return _attend(kv[0], None, q[0])[0].cpu().numpy(), _weigh(w[0], kv[1]).cpu().numpy()
    out = torch.empty(q.shape, dtype=torch.float64, device="cuda")
    for s in range(case["seqs"]):
        for i in range(case["layers"]):
            kv = [_quantized(torch.cat([xs[s][i, j], new[s, i, j]], 1)) for j in (0, 1)]
            out[i, s] = _attend(kv[0], kv[1], q[i, s])[1]
        xs[s] = None
    return out
