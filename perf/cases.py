"""What a model built on this engine has it do, as single calls and short
call sequences through the package's public entry points.

The shapes are those of the reference's graphs: the Qwen3 LM (0.6B: 16 query
heads over 8 KV heads, 28 layers; 4B: 32 over 8) with its prompt, its KV-cache
writes and its decode steps, the condition encoders (16 over 8), and the DiT
(16 over 8) with its full, sliding-window and cross-attention layers, where
the number of tokens follows from the song's length and is seldom round.

Every case is a dict of plain values with a "kind" (see the tables of
functions at the end); sequence lengths and paddings are texts of whole
numbers.  Tensors lie in memory as the reference lays them out.
"""
from __future__ import annotations

import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.abspath("acestep.cpp_amd"))
import mxfa  # noqa: E402

D = 128
SCALE = 1.0 / math.sqrt(D)
F32, F16, Q8_0, I32, I64, BF16 = 0, 1, 8, 26, 27, 30
TYPES = {"f16": (F16, torch.float16), "bf16": (BF16, torch.bfloat16)}
Q8_ROW = D // 32 * 34
EPS, FREQ_BASE = 1e-6, 1e6


def listed():
    return [
        # One attention call of a single-sequence decode step, the smallest
        # call there is: one token of the 0.6B LM, 411 keys in a window of 512.
        dict(name="decode_one", kind="decode", Nh=16, Nkv=8, lens="411", max_seq=2048, kv="f16"),
        # A whole decode token of the 0.6B LM with classifier-free guidance
        # (two sequences), replayed as a HIP graph: per layer both KV-cache
        # writes and the attention call.
        dict(name="decode_token", kind="token", Nh=16, Nkv=8, layers=28, lens="1377,1290", max_seq=2048),
        # Batched CFG decode of the 4B LM: four songs, eight sequences of
        # ragged length over one cache.
        dict(name="decode_batch", kind="decode", Nh=32, Nkv=8, lens="7340,2218,4975,1180,7302,2190,4961,1163",
             max_seq=8192, kv="f16"),
        # The same over a quantised cache at full context.
        dict(name="decode_q8", kind="decode", Nh=32, Nkv=8, lens="8192,8192,8192,8192", max_seq=8192, kv="q8_0"),
        # A 2048-token causal prompt of the 4B LM into an empty cache.
        dict(name="prompt", kind="prompt", Nh=32, Nkv=8, tokens=2048, pos=0, max_seq=2048, kv="f16"),
        # One layer's attention for the next piece of a prompt: the
        # pre-attention step (norms, RoPE, casts, cache rows) and attention
        # on the 16-bit Q it leaves, the causal mask as metadata.
        dict(name="prompt_piece", kind="layer", Nh=32, Nkv=8, tokens=333, pos=1800, max_seq=4096, kv="f16"),
        # A prompt continued over a quantised cache: both cache writes, then
        # attention.
        dict(name="prompt_q8", kind="prompt_q8", Nh=32, Nkv=8, tokens=1000, pos=500, max_seq=4096),
        # The lyric encoder's eight layers, window mask on the even ones and
        # none on the odd ones, inside one graph bracket.
        dict(name="encoder", kind="encoder", Nh=16, Nkv=8, tokens=437, layers=8, mask="window", window=128),
        # Full self-attention of the DiT, four minutes of audio, CFG pair.
        dict(name="dit_self", kind="dit_self", Nh=16, Nkv=8, tokens=3000, batch=2, kv="f16"),
        # The same for 87 seconds in bfloat16.
        dict(name="dit_self_bf16", kind="dit_self", Nh=16, Nkv=8, tokens=1085, batch=2, kv="bf16"),
        # The DiT's sliding-window layer under its dense mask, 87 seconds.
        dict(name="dit_window", kind="dit_window", Nh=16, Nkv=8, tokens=1085, batch=2, window=128, kv="f16"),
        # The DiT's cross-attention over 238 encoder tokens, some of them
        # padding, under its dense mask.
        dict(name="dit_cross", kind="dit_cross", Nh=16, Nkv=8, tokens=1085, batch=2, enc=238, pads="31,31", kv="f16"),
    ]


def _log_int(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["decode", "token", "prompt", "layer", "prompt_q8", "encoder", "dit_self", "dit_window",
                       "dit_cross"])
    Nh = rng.choice([16, 32])
    kv = rng.choice(["f16", "f16", "bf16"])
    if kind == "decode":
        kv = rng.choice(["f16", "bf16", "q8_0"])
        top = _log_int(rng, 64, 8192)
        n = rng.choice([1, 2, 4, 8])
        lens = [top] + [_log_int(rng, max(16, top // 8), top) for _ in range(n - 1)]
        return dict(kind=kind, Nh=Nh, Nkv=8, lens=",".join(map(str, lens)), max_seq=8192, kv=kv)
    if kind == "token":
        n = rng.choice([1, 2, 4])
        top = _log_int(rng, 64, 4096 // n)
        lens = [top] + [_log_int(rng, max(16, top // 4), top) for _ in range(n - 1)]
        return dict(kind=kind, Nh=Nh, Nkv=8, layers=28 if Nh == 16 else 36, lens=",".join(map(str, lens)),
                    max_seq=-(-top // 256) * 256)
    if kind in ("prompt", "layer"):
        return dict(kind=kind, Nh=Nh, Nkv=8, tokens=_log_int(rng, 20, 2048), pos=rng.choice([0, rng.randint(1, 4000)]),
                    max_seq=8192, kv=kv)
    if kind == "prompt_q8":
        return dict(kind=kind, Nh=Nh, Nkv=8, tokens=_log_int(rng, 20, 1500), pos=rng.randint(0, 2500), max_seq=4096)
    if kind == "encoder":
        if rng.random() < 0.5:   # the text encoder: causal, every layer
            return dict(kind=kind, Nh=16, Nkv=8, tokens=_log_int(rng, 20, 512), layers=28, mask="causal", window=0)
        return dict(kind=kind, Nh=16, Nkv=8, tokens=_log_int(rng, 50, 1200), layers=8, mask="window", window=128)
    batch = rng.choice([1, 2, 4])
    top = int(3000 * math.sqrt(2 / max(batch, 2)))
    c = dict(kind=kind, Nh=16, Nkv=8, tokens=_log_int(rng, 125, top), batch=batch)
    if kind == "dit_window":
        c["window"] = 128
    if kind == "dit_cross":
        c["enc"] = _log_int(rng, 40, 512)
        p = [rng.randint(0, c["enc"] // 2) for _ in range(max(batch // 2, 1))]
        c["pads"] = ",".join(map(str, (p + p)[:batch]))
    c["kv"] = kv
    return c


# -- helpers -------------------------------------------------------------------


def _ints(text):
    return [int(x) for x in text.split(",")]


def _window(n, max_seq):
    """The cache window a step reads: its length rounded up to 256 keys."""
    return min(-(-n // 256) * 256, max_seq)


def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _normal(g, *shape, dtype=torch.float32):
    x = torch.randn(*shape, generator=g, device="cuda", dtype=torch.float32)
    return x if dtype == torch.float32 else x.to(dtype)


def _view(t, type_, ne, nb, offset=0):
    return mxfa.DeviceView(type_, tuple(ne), tuple(nb), t.data_ptr() + offset, t)


def _out(B, S, Nh):
    o = torch.empty(B, S, Nh, D, dtype=torch.float32, device="cuda")
    return o, _view(o, F32, (D, Nh, S, B), (4, 4 * D, 4 * D * Nh, 4 * D * Nh * S))


def _q_rows(q, B, S, Nh, size=4, type_=F32):
    """Q as the projection leaves it, [B, S, Nh, D], seen as [D, S, Nh, B]."""
    return _view(q, type_, (D, S, Nh, B), (size, size * D * Nh, size * D, size * D * Nh * S))


def _cache_view(t, type_, window, Nkv, B, max_seq):
    row = 2 * D if type_ != Q8_0 else Q8_ROW
    return _view(t, type_, (D, window, Nkv, B), (2 if type_ != Q8_0 else 34, row, row * max_seq, row * max_seq * Nkv))


def _mask_view(live):
    """live: bool [B, Sq, Skv] -> the F16 mask tensor (0 / -inf) and its view."""
    m = torch.zeros(live.shape, dtype=torch.float16, device="cuda").masked_fill_(~live, float("-inf"))
    B, Sq, Skv = live.shape
    return m, _view(m, F16, (Skv, Sq, 1, B), (2, 2 * Skv, 2 * Skv * Sq, 2 * Skv * Sq))


def _q8_np(x):
    """Q8_0 blocks of float32 rows of 128 (ggml's layout and rounding): the
    bytes, and the values they stand for in 64 bits."""
    xb = np.asarray(x, dtype=np.float32).reshape(-1, 32)
    amax = np.abs(xb).max(axis=1)
    d = amax / np.float32(127.0)
    inv = np.divide(np.float32(127.0), amax, out=np.zeros_like(amax), where=amax != 0)
    q = np.rint(xb * inv[:, None]).astype(np.int8)
    d16 = d.astype(np.float16)
    out = np.empty((xb.shape[0], 34), dtype=np.uint8)
    out[:, :2] = d16.view(np.uint8).reshape(-1, 2)
    out[:, 2:] = q.view(np.uint8)
    return out.reshape(-1), (q.astype(np.float64) * d16.astype(np.float64)[:, None]).reshape(np.shape(x))


def _q8_pack(x):
    """The same blocks made on the GPU (inputs only: whatever bytes come out
    are the cache's contents)."""
    xb = x.reshape(-1, 32)
    amax = xb.abs().amax(dim=1, keepdim=True)
    q = torch.round(xb * (127.0 / amax)).to(torch.int8)
    d = (amax / 127.0).to(torch.float16)
    return torch.cat([d.view(torch.uint8), q.view(torch.uint8)], dim=1).reshape(-1)


def _q8_values(b):
    """The values of Q8_0 bytes, in 64 bits."""
    b = b.reshape(-1, 34)
    d = b[:, :2].contiguous().view(torch.float16).double()
    return (b[:, 2:].contiguous().view(torch.int8).double() * d).reshape(-1)


def _attend(q, k, v, live):
    """Softmax attention in 64 bits.  q [B, S, Nh, D], k / v [B, Nkv, Skv, D],
    live: None, or bool [B or 1, S, Skv]; a query with no live key gives 0."""
    B, S, Nh, _ = q.shape
    Nkv = k.shape[1]
    out = torch.empty(B, S, Nh, D, dtype=torch.float64, device=q.device)
    for b in range(B):
        dead = None if live is None else ~live[b % live.shape[0]]
        for h in range(Nh):
            kh, vh = k[b, h // (Nh // Nkv)].double(), v[b, h // (Nh // Nkv)].double()
            s = (q[b, :, h].double() @ kh.t().contiguous()) * SCALE
            if dead is not None:
                s.masked_fill_(dead, float("-inf"))
            out[b, :, h] = torch.nan_to_num(torch.softmax(s, dim=-1)) @ vh
    return out


def _causal(S, Skv, pos):
    return (torch.arange(Skv, device="cuda")[None, :] <= pos + torch.arange(S, device="cuda")[:, None])[None]


def _band(S, window):
    i = torch.arange(S, device="cuda")
    return ((i[:, None] - i[None, :]).abs() <= (window if S > window else S))[None]


def _lengths(lens, Skv):
    n = torch.tensor(lens, device="cuda")
    return torch.arange(Skv, device="cuda")[None, None, :] < n[:, None, None]


def _pairs_causal(S, pos):
    return S * pos + S * (S + 1) // 2


def _pairs_band(S, window):
    if S <= window:
        return S * S
    return S * (2 * window + 1) - window * (window + 1)


def _attention_work(c, queries, pairs, kv_rows, mask_values, q_bytes=4, kv_row=2 * D):
    """queries: (query, head) rows; pairs: unmasked (query, key) pairs over
    all heads; kv_rows: live K rows over all KV heads and batches."""
    return dict(bytes=queries * D * (q_bytes + 4) + 2 * kv_rows * kv_row + 2 * mask_values, flops=4 * D * pairs)


# -- decode: one token per sequence ----------------------------------------------


def _decode_inputs(c, seed):
    lens = _ints(c["lens"])
    N, Nh, Nkv, M = len(lens), c["Nh"], c["Nkv"], c["max_seq"]
    g = _gen(seed)
    q = _normal(g, N, 1, Nh, D)
    if c["kv"] == "q8_0":
        k, v = (_q8_pack(_normal(g, N * Nkv * M, D)) for _ in range(2))
    else:
        k, v = (_normal(g, N, Nkv, M, D, dtype=TYPES[c["kv"]][1]) for _ in range(2))
    return lens, q, k, v


def _decode_prepare(c, seed):
    lens, q, k, v = _decode_inputs(c, seed)
    N, Nh, Nkv, M = len(lens), c["Nh"], c["Nkv"], c["max_seq"]
    w = _window(max(lens), M)
    t = Q8_0 if c["kv"] == "q8_0" else TYPES[c["kv"]][0]
    m, mv = _mask_view(_lengths(lens, w))
    o, ov = _out(N, 1, Nh)
    return dict(kind="attend", out=o, dst=ov, mask=mv, k=_cache_view(k, t, w, Nkv, N, M), v=_cache_view(v, t, w, Nkv, N, M),
                q=_view(q, F32, (D, 1, Nh, N), (4, 4 * D, 4 * D, 4 * D * Nh)))


def _attend_run(s):
    mxfa.flash_attn_ext(s["q"], s["k"], s["v"], s["mask"], SCALE, dst=s["dst"])
    return s["out"]


def _decode_exact(c, seed):
    lens, q, k, v = _decode_inputs(c, seed)
    N, Nkv, M = len(lens), c["Nkv"], c["max_seq"]
    w = _window(max(lens), M)
    if c["kv"] == "q8_0":
        q = torch.from_numpy(_q8_np(q.cpu().numpy())[1]).cuda()
        k, v = (_q8_values(x).reshape(N, Nkv, M, D) for x in (k, v))
    else:
        q = q.to(TYPES[c["kv"]][1])
    return _attend(q, k[:, :, :w], v[:, :, :w], _lengths(lens, w))


def _decode_work(c):
    lens = _ints(c["lens"])
    w = _window(max(lens), c["max_seq"])
    return _attention_work(c, len(lens) * c["Nh"], sum(lens) * c["Nh"], sum(lens) * c["Nkv"], len(lens) * w,
                           kv_row=Q8_ROW if c["kv"] == "q8_0" else 2 * D)


# -- a decode token of the whole LM: every layer's cache writes and attention ----


def _token_inputs(c, seed):
    lens = _ints(c["lens"])
    N, Nh, Nkv, M, L = len(lens), c["Nh"], c["Nkv"], c["max_seq"], c["layers"]
    g = _gen(seed)
    q = _normal(g, L, N, 1, Nh, D)
    new = _normal(g, 2, L, N, Nkv, D)
    cache = torch.empty(2, L, N, Nkv, M, D, dtype=torch.float16, device="cuda")
    for x in cache.reshape(2 * L, -1):
        x.copy_(torch.randn(x.numel(), generator=g, device="cuda"))
    return lens, q, new, cache


def _token_prepare(c, seed):
    lens, q, new, cache = _token_inputs(c, seed)
    N, Nh, Nkv, M, L = len(lens), c["Nh"], c["Nkv"], c["max_seq"], c["layers"]
    w = _window(max(lens), M)
    m, mv = _mask_view(_lengths(lens, w))
    out = torch.empty(L, N, 1, Nh, D, dtype=torch.float32, device="cuda")
    ids = torch.tensor([n - 1 for n in lens], dtype=torch.int64, device="cuda")
    iv = _view(ids, I64, (1, 1, N, 1), (8, 8, 8, 8 * N))
    calls = []
    for i in range(L):
        rows = [_view(new[j, i], F32, (D, 1, Nkv, N), (4, 4 * D, 4 * D, 4 * D * Nkv)) for j in range(2)]
        full = [_cache_view(cache[j, i], F16, M, Nkv, N, M) for j in range(2)]
        kv = [_cache_view(cache[j, i], F16, w, Nkv, N, M) for j in range(2)]
        qv = _view(q[i], F32, (D, 1, Nh, N), (4, 4 * D, 4 * D, 4 * D * Nh))
        ov = _view(out[i], F32, (D, Nh, 1, N), (4, 4 * D, 4 * D * Nh, 4 * D * Nh))
        calls.append((rows, full, kv, qv, ov))

    def token():
        for rows, full, kv, qv, ov in calls:
            mxfa.set_rows(full[0], rows[0], iv)
            mxfa.set_rows(full[1], rows[1], iv)
            mxfa.flash_attn_ext(qv, kv[0], kv[1], mv, SCALE, dst=ov)

    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):   # sizes the stream's workspace
        token()
    torch.cuda.current_stream().wait_stream(side)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=side):
        token()
    return dict(kind="token", graph=graph, out=out, cache=cache, keep=(q, new, m, ids, calls, side))


def _token_run(s):
    s["graph"].replay()
    return [s["out"], s["cache"]]


def _token_exact(c, seed):
    lens, q, new, cache = _token_inputs(c, seed)
    w = _window(max(lens), c["max_seq"])
    out = []
    for b, n in enumerate(lens):
        cache[:, :, b, :, n - 1] = new[:, :, b].half()
    for i in range(c["layers"]):
        out.append(_attend(q[i].half(), cache[0, i, :, :, :w], cache[1, i, :, :, :w], _lengths(lens, w)))
    # (the written rows are whatever rounding to 16 bits gives; the rest of
    # the cache is the input's)
    return [torch.stack(out), cache]


def _token_work(c):
    lens = _ints(c["lens"])
    w = _window(max(lens), c["max_seq"])
    a = _attention_work(c, len(lens) * c["Nh"], sum(lens) * c["Nh"], sum(lens) * c["Nkv"], 0)
    rows = 2 * len(lens) * c["Nkv"] * D * (4 + 2)
    return dict(bytes=c["layers"] * (a["bytes"] + rows) + 2 * len(lens) * w, flops=c["layers"] * a["flops"])


# -- a causal prompt over a 16-bit cache ------------------------------------------


def _prompt_inputs(c, seed):
    dt = TYPES[c["kv"]][1]
    g = _gen(seed)
    q = _normal(g, 1, c["tokens"], c["Nh"], D)
    k, v = (_normal(g, 1, c["Nkv"], c["max_seq"], D, dtype=dt) for _ in range(2))
    return q, k, v


def _prompt_prepare(c, seed):
    q, k, v = _prompt_inputs(c, seed)
    S, Nh, Nkv, M = c["tokens"], c["Nh"], c["Nkv"], c["max_seq"]
    w = _window(c["pos"] + S, M)
    t = TYPES[c["kv"]][0]
    m, mv = _mask_view(_causal(S, w, c["pos"]))
    o, ov = _out(1, S, Nh)
    return dict(kind="attend", out=o, dst=ov, mask=mv, q=_q_rows(q, 1, S, Nh), k=_cache_view(k, t, w, Nkv, 1, M),
                v=_cache_view(v, t, w, Nkv, 1, M))


def _prompt_exact(c, seed):
    q, k, v = _prompt_inputs(c, seed)
    n = c["pos"] + c["tokens"]
    return _attend(q.to(k.dtype), k[:, :, :n], v[:, :, :n], _causal(c["tokens"], n, c["pos"]))


def _prompt_work(c):
    S, pos = c["tokens"], c["pos"]
    return _attention_work(c, S * c["Nh"], _pairs_causal(S, pos) * c["Nh"], (S + pos) * c["Nkv"],
                           S * _window(pos + S, c["max_seq"]))


# -- one layer of a prompt's next piece: pre-attention step, attention -----------


def _layer_inputs(c, seed):
    S, Nh, Nkv, M = c["tokens"], c["Nh"], c["Nkv"], c["max_seq"]
    dt = TYPES[c["kv"]][1]
    g = _gen(seed)
    x = 2.0 * _normal(g, S, Nh + 2 * Nkv, D)
    w = 1.0 + 0.2 * _normal(g, 2, D)
    cache = _normal(g, 2, Nkv, M, D, dtype=dt)
    return x, w, cache


def _layer_prepare(c, seed):
    x, w, cache = _layer_inputs(c, seed)
    S, Nh, Nkv, M, pos = c["tokens"], c["Nh"], c["Nkv"], c["max_seq"], c["pos"]
    t, dt = TYPES[c["kv"]]
    H = Nh + 2 * Nkv
    nb = (4, 4 * D, 4 * D * H, 4 * D * H * S)
    p = torch.arange(pos, pos + S, dtype=torch.int32, device="cuda")
    rows = p.to(torch.int64)
    qo = torch.empty(S, Nh, D, dtype=dt, device="cuda")
    o, ov = _out(1, S, Nh)
    n = pos + S
    wnb = (4, 4 * D, 4 * D, 4 * D)
    return dict(
        kind="layer", out=[qo, cache, o], dst=ov, spec=mxfa.mask_spec(causal=True, pos0=pos),
        x=[_view(x, F32, (D, Nh, S, 1), nb), _view(x, F32, (D, Nkv, S, 1), nb, 4 * D * Nh),
           _view(x, F32, (D, Nkv, S, 1), nb, 4 * D * (Nh + Nkv))],
        w=[_view(w, F32, (D, 1, 1, 1), wnb, 4 * D * j) for j in range(2)],
        pos=_view(p, I32, (S, 1, 1, 1), (4, 4 * S, 4 * S, 4 * S)),
        rows=_view(rows, I64, (S, 1, 1, 1), (8, 8 * S, 8 * S, 8 * S)),
        q_out=_view(qo, t, (D, Nh, S, 1), (2, 2 * D, 2 * D * Nh, 2 * D * Nh * S)),
        caches=[_cache_view(cache[j], t, M, Nkv, 1, M) for j in range(2)],
        q=_q_rows(qo, 1, S, Nh, 2, t), k=_cache_view(cache[0], t, n, Nkv, 1, M), v=_cache_view(cache[1], t, n, Nkv, 1, M))


def _layer_run(s):
    mxfa.qk_norm_rope(*s["x"], *s["w"], s["pos"], EPS, FREQ_BASE, s["q_out"], *s["caches"], s["rows"])
    mxfa.flash_attn_ext_masked(s["q"], s["k"], s["v"], s["spec"], SCALE, dst=s["dst"])
    return s["out"]


def _layer_exact(c, seed):
    x, w, cache = _layer_inputs(c, seed)
    S, Nh, Nkv, pos = c["tokens"], c["Nh"], c["Nkv"], c["pos"]
    # the angle of pair i is i float multiplications of the position (the
    # RoPE's definition in ggml); its sine and cosine are taken in 64 bits
    scale = torch.tensor(FREQ_BASE, dtype=torch.float32).pow(-2.0 / D).cuda()
    a = torch.arange(pos, pos + S, device="cuda").float()
    angles = []
    for _ in range(D // 2):
        angles.append(a)
        a = a * scale
    angles = torch.stack(angles, dim=-1).double()[:, None]
    x, w = x.double(), w.double()

    def turned(y, weight):
        y = y / torch.sqrt(y.square().mean(dim=-1, keepdim=True) + EPS) * weight
        lo, hi = y[..., :D // 2], y[..., D // 2:]
        return torch.cat([lo * angles.cos() - hi * angles.sin(), lo * angles.sin() + hi * angles.cos()], dim=-1)

    q, k, v = turned(x[:, :Nh], w[0]), turned(x[:, Nh:Nh + Nkv], w[1]), x[:, Nh + Nkv:]
    dt = cache.dtype
    cache[0, :, pos:pos + S] = k.transpose(0, 1).to(dt)
    cache[1, :, pos:pos + S] = v.transpose(0, 1).to(dt)
    n = pos + S
    o = _attend(q.to(dt)[None], cache[0:1, :, :n], cache[1:2, :, :n], _causal(S, n, pos))
    return [q, cache, o]


def _layer_work(c):
    S, pos, rows = c["tokens"], c["pos"], c["tokens"] * (c["Nh"] + 2 * c["Nkv"])
    a = _attention_work(c, S * c["Nh"], _pairs_causal(S, pos) * c["Nh"], (S + pos) * c["Nkv"], 0, q_bytes=2)
    return dict(bytes=a["bytes"] + rows * D * (4 + 2) + S * 12, flops=a["flops"])


# -- a prompt over a quantised cache: cache writes, attention ---------------------


def _prompt_q8_inputs(c, seed):
    S, Nh, Nkv, M = c["tokens"], c["Nh"], c["Nkv"], c["max_seq"]
    g = _gen(seed)
    q = _normal(g, 1, S, Nh, D)
    new = _normal(g, 2, Nkv, S, D)
    cache = torch.stack([_q8_pack(_normal(g, Nkv * M, D)) for _ in range(2)])
    return q, new, cache


def _prompt_q8_prepare(c, seed):
    q, new, cache = _prompt_q8_inputs(c, seed)
    S, Nh, Nkv, M, pos = c["tokens"], c["Nh"], c["Nkv"], c["max_seq"], c["pos"]
    w = _window(pos + S, M)
    m, mv = _mask_view(_causal(S, w, pos))
    o, ov = _out(1, S, Nh)
    ids = torch.arange(pos, pos + S, dtype=torch.int64, device="cuda")
    return dict(kind="prompt_q8", out=[o, cache], dst=ov, mask=mv, q=_q_rows(q, 1, S, Nh),
                new=[_view(new[j], F32, (D, S, Nkv, 1), (4, 4 * D, 4 * D * S, 4 * D * S * Nkv)) for j in range(2)],
                ids=_view(ids, I64, (S, 1, 1, 1), (8, 8 * S, 8 * S, 8 * S)),
                full=[_cache_view(cache[j], Q8_0, M, Nkv, 1, M) for j in range(2)],
                kv=[_cache_view(cache[j], Q8_0, w, Nkv, 1, M) for j in range(2)])


def _prompt_q8_run(s):
    for j in range(2):
        mxfa.set_rows(s["full"][j], s["new"][j], s["ids"])
    mxfa.flash_attn_ext(s["q"], s["kv"][0], s["kv"][1], s["mask"], SCALE, dst=s["dst"])
    return s["out"]


def _prompt_q8_exact(c, seed):
    q, new, cache = _prompt_q8_inputs(c, seed)
    S, Nkv, M, pos = c["tokens"], c["Nkv"], c["max_seq"], c["pos"]
    kv = []
    for j in range(2):
        x = _q8_values(cache[j]).reshape(Nkv, M, D)
        x[:, pos:pos + S] = torch.from_numpy(_q8_np(new[j].cpu().numpy())[1]).cuda()
        kv.append(x[None, :, :pos + S])
    q = torch.from_numpy(_q8_np(q.cpu().numpy())[1]).cuda()
    return [_attend(q, kv[0], kv[1], _causal(S, pos + S, pos)), None]


def _prompt_q8_work(c):
    S, pos = c["tokens"], c["pos"]
    a = _attention_work(c, S * c["Nh"], _pairs_causal(S, pos) * c["Nh"], (S + pos) * c["Nkv"],
                        S * _window(pos + S, c["max_seq"]), kv_row=Q8_ROW)
    return dict(bytes=a["bytes"] + 2 * S * c["Nkv"] * (4 * D + Q8_ROW) + 8 * S, flops=a["flops"])


# -- an encoder's layers: contiguous K / V, one mask tensor for all of them -------


def _encoder_inputs(c, seed):
    S, Nh, Nkv, L = c["tokens"], c["Nh"], c["Nkv"], c["layers"]
    g = _gen(seed)
    q = _normal(g, L, 1, S, Nh, D)
    kv = _normal(g, 2, L, 1, Nkv, S, D, dtype=torch.float16)
    return q, kv, (_causal(S, S, 0) if c["mask"] == "causal" else _band(S, c["window"]))


def _encoder_masked(c, i):
    """Causal encoders mask every layer, windowed ones the even layers."""
    return c["mask"] == "causal" or i % 2 == 0


def _encoder_prepare(c, seed):
    q, kv, live = _encoder_inputs(c, seed)
    S, Nh, Nkv, L = c["tokens"], c["Nh"], c["Nkv"], c["layers"]
    m, mv = _mask_view(live)
    out = torch.empty(L, 1, S, Nh, D, dtype=torch.float32, device="cuda")
    calls = []
    for i in range(L):
        k, v = (_cache_view(kv[j, i], F16, S, Nkv, 1, S) for j in range(2))
        ov = _view(out[i], F32, (D, Nh, S, 1), (4, 4 * D, 4 * D * Nh, 4 * D * Nh * S))
        calls.append((_q_rows(q[i], 1, S, Nh), k, v, mv if _encoder_masked(c, i) else None, ov))
    return dict(kind="encoder", out=out, calls=calls, keep=(q, kv, m))


def _encoder_run(s):
    with mxfa.graph():
        for q, k, v, m, o in s["calls"]:
            mxfa.flash_attn_ext(q, k, v, m, SCALE, dst=o)
    return s["out"]


def _encoder_exact(c, seed):
    q, kv, live = _encoder_inputs(c, seed)
    return torch.stack([_attend(q[i].half(), kv[0, i], kv[1, i], live if _encoder_masked(c, i) else None)
                        for i in range(c["layers"])])


def _encoder_work(c):
    S, n = c["tokens"], dict(bytes=2 * c["tokens"] ** 2, flops=0)
    for i in range(c["layers"]):
        pairs = S * S
        if _encoder_masked(c, i):
            pairs = _pairs_causal(S, 0) if c["mask"] == "causal" else _pairs_band(S, c["window"])
        a = _attention_work(c, S * c["Nh"], pairs * c["Nh"], S * c["Nkv"], 0)
        n = dict(bytes=n["bytes"] + a["bytes"], flops=n["flops"] + a["flops"])
    return n


# -- the DiT's attention -----------------------------------------------------------


def _dit_inputs(c, seed):
    S, Nh, Nkv, B = c["tokens"], c["Nh"], c["Nkv"], c["batch"]
    g = _gen(seed)
    cross = c["kind"] == "dit_cross"
    q = _normal(g, B, Nh, S, D) if cross else _normal(g, B, S, Nh, D)
    k, v = (_normal(g, B, Nkv, c["enc"] if cross else S, D, dtype=TYPES[c["kv"]][1]) for _ in range(2))
    live = None
    if cross:
        live = _lengths([c["enc"] - p for p in _ints(c["pads"])], c["enc"]).expand(B, S, c["enc"])
    elif c["kind"] == "dit_window":
        live = _band(S, c["window"]).expand(B, S, S)
    return q, k, v, live


def _dit_prepare(c, seed):
    q, k, v, live = _dit_inputs(c, seed)
    S, Nh, Nkv, B = c["tokens"], c["Nh"], c["Nkv"], c["batch"]
    Skv, t = k.shape[2], TYPES[c["kv"]][0]
    m, mv = _mask_view(live) if live is not None else (None, None)
    o, ov = _out(B, S, Nh)
    # cross-attention's Q is contiguous [D, S, Nh, B] (its norm's result)
    qv = _view(q, F32, (D, S, Nh, B), (4, 4 * D, 4 * D * S, 4 * D * S * Nh)) if c["kind"] == "dit_cross" \
        else _q_rows(q, B, S, Nh)
    return dict(kind="attend", out=o, dst=ov, mask=mv, q=qv, k=_cache_view(k, t, Skv, Nkv, B, Skv),
                v=_cache_view(v, t, Skv, Nkv, B, Skv))


def _dit_exact(c, seed):
    q, k, v, live = _dit_inputs(c, seed)
    if c["kind"] == "dit_cross":
        q = q.transpose(1, 2)
    return _attend(q.to(k.dtype), k, v, live)


def _dit_work(c):
    S, B = c["tokens"], c["batch"]
    if c["kind"] == "dit_cross":
        rows = sum(c["enc"] - p for p in _ints(c["pads"]))
        return _attention_work(c, S * B * c["Nh"], rows * S * c["Nh"], rows * c["Nkv"], S * c["enc"] * B)
    pairs = S * S if c["kind"] == "dit_self" else _pairs_band(S, c["window"])
    return _attention_work(c, S * B * c["Nh"], pairs * B * c["Nh"], S * B * c["Nkv"],
                           0 if c["kind"] == "dit_self" else S * S * B)


# -- the interface -----------------------------------------------------------------

_DIT = (_dit_prepare, _dit_exact, _dit_work)
_KINDS = {
    "decode": (_decode_prepare, _decode_exact, _decode_work),
    "token": (_token_prepare, _token_exact, _token_work),
    "prompt": (_prompt_prepare, _prompt_exact, _prompt_work),
    "layer": (_layer_prepare, _layer_exact, _layer_work),
    "prompt_q8": (_prompt_q8_prepare, _prompt_q8_exact, _prompt_q8_work),
    "encoder": (_encoder_prepare, _encoder_exact, _encoder_work),
    "dit_self": _DIT, "dit_window": _DIT, "dit_cross": _DIT,
}
_RUNS = {"attend": _attend_run, "token": _token_run, "layer": _layer_run, "prompt_q8": _prompt_q8_run,
         "encoder": _encoder_run}


def prepare(case, seed):
    return _KINDS[case["kind"]][0](case, seed)


def run(state):
    return _RUNS[state["kind"]](state)


def exact(case, seed):
    return _KINDS[case["kind"]][1](case, seed)


def work(case):
    return _KINDS[case["kind"]][2](case)


def tolerance(case):
    # float16 attention rounds the probabilities to 11 bits before the
    # second product, relative to a running maximum that depends on how the
    # keys are split: it lies 1.3e-4 to 2.1e-4 of its norm from the 64-bit
    # result, so two correct results differ by up to about 3e-4 (largest: a
    # causal prompt's first rows, 5e-4 where the root mean square is 0.08).
    if case["kind"] == "prompt_q8":   # both factors of a product rounded once: 4.2e-4
        return {"rel": 2e-3, "max": 3e-2}
    if case.get("kv") == "bf16":
        # probabilities carried as two bfloat16 parts: 2.4e-6 from 64 bits;
        # the pre-attention step's own outputs are rounded to 8 bits, and a
        # value on the edge between two may fall either way
        return {"rel": 1e-3, "max": 2e-2} if case["kind"] == "layer" else {"rel": 2e-5, "max": 1e-3}
    return {"rel": 1e-3, "max": 2e-2}
