"""Performance cases of the paged KV-cache path: decode steps, chunked prefill,
the O-projection and the gather back to the host's cache layout, each through
the package's public entry points.

listed() names the cases, draw(rng) makes further ones of the same ranges,
prepare / run make one case's state and one pass over it, work() counts the
bytes and operations a pass cannot do without, exact() is the pass in float64
by plain torch, tolerance() how far a correct implementation may be from it.

Shapes are the ones bench.py names: TinyLlama-1.1B (32 query / 4 kv heads of
64), Llama-3-8B (32 / 8 of 128) and Llama-3-70B (64 / 8 of 128).
"""
import importlib
import math

import numpy as np
import torch

gi = importlib.import_module("go-infer_amd")

KV = {"f32": gi.KV_F32, "f16": gi.KV_F16, "q8_0": gi.KV_Q8_0, "q4_0": gi.KV_Q4_0}
WT = {"f32": gi.GGML_F32, "f16": gi.GGML_F16, "q4_0": gi.GGML_Q4_0, "q8_0": gi.GGML_Q8_0}
KV_BYTES = {"f32": 4.0, "f16": 2.0, "q8_0": 34 / 32, "q4_0": 18 / 32}  # per stored element
SHAPES = {"tinyllama": dict(heads=32, kv_heads=4, hd=64, theta=10000.0),
          "llama8b": dict(heads=32, kv_heads=8, hd=128, theta=500000.0),
          "llama70b": dict(heads=64, kv_heads=8, hd=128, theta=500000.0)}


def _decode(shape, kv, batch, lo, hi, layers, rope, page):
    return dict(kind="decode", shape=shape, kv=kv, batch=batch, ctx_lo=lo, ctx_hi=hi, layers=layers, rope=rope,
                page=page)


def _prefill(shape, kv, batch, start, prompt, chunk, rope, page):
    return dict(kind="prefill", shape=shape, kv=kv, batch=batch, start=start, prompt=prompt, chunk=chunk, rope=rope,
                page=page)


def _matmul(wtype, rows, cols, batch, layers):
    return dict(kind="matmul", wtype=wtype, rows=rows, cols=cols, batch=batch, layers=layers)


def _get(shape, kv, tokens, widen, page):
    return dict(kind="get", shape=shape, kv=kv, tokens=tokens, widen=widen, page=page)


def listed():
    cases = {
        # one token of the reference's CPU-runnable case: a single short
        # TinyLlama chat, every layer's store + attention (launches count)
        "decode_tinyllama_b1_f32": _decode("tinyllama", "f32", 1, 197, 197, 22, False, 16),
        # one user in a long Llama-3-8B conversation: RoPE + store + attention
        # of the first eight layers of a token
        "decode_llama8b_b1_f16_long": _decode("llama8b", "f16", 1, 6001, 6001, 8, True, 16),
        # a small server: 32 conversations of all lengths, one layer
        "decode_llama8b_b32_f16_ragged": _decode("llama8b", "f16", 32, 512, 4096, 1, True, 16),
        # a few very long documents on the largest model, one layer
        "decode_llama70b_b8_f16_32k": _decode("llama70b", "f16", 8, 32768, 32768, 1, False, 32),
        # a mid-size server that keeps its cache in four bits, one layer
        "decode_llama8b_b48_q4": _decode("llama8b", "q4_0", 48, 1500, 6500, 1, True, 16),
        # a full server near its context limit with an 8-bit cache, one layer
        "decode_llama8b_b256_q8_8k": _decode("llama8b", "q8_0", 256, 6144, 8192, 1, False, 16),
        # one user's prompt of odd length in 512-token chunks, one layer
        "prefill_llama8b_b1_f16": _prefill("llama8b", "f16", 1, 0, 2300, 512, True, 16),
        # four full prompts over an 8-bit cache in 512-token chunks, one layer
        "prefill_llama8b_b4_q8_4k": _prefill("llama8b", "q8_0", 4, 0, 4096, 512, False, 16),
        # a short TinyLlama prompt in one chunk over the default f32 cache
        "prefill_tinyllama_b1_f32": _prefill("tinyllama", "f32", 1, 0, 300, 300, True, 16),
        # the O-projections of one token, all 32 layers, 4-bit weights
        "oproj_llama8b_b1_q4": _matmul("q4_0", 4096, 4096, 1, 32),
        # the O-projection of a large running batch, 8-bit weights
        "oproj_llama8b_b256_q8": _matmul("q8_0", 4096, 4096, 256, 4),
        # a cached conversation handed to the host's contiguous cache layout
        # (KVCache.Get / ForkAt) as stored halves, one layer
        "get_llama8b_f16": _get("llama8b", "f16", 6001, False, 16),
    }
    return [dict(c, name=n) for n, c in cases.items()]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case: any model shape, cache and weight type, page size and
    size, sizes spread over their logarithm, within the largest listed
    case's cost."""
    kind = rng.choice(("decode", "decode", "decode", "prefill", "prefill", "matmul", "matmul", "get"))
    shape = rng.choice(sorted(SHAPES))
    S = SHAPES[shape]
    kv = rng.choice(sorted(KV))
    page = rng.choice((16, 32))
    if kind == "decode":
        batch = _log_int(rng, 1, 256)
        hi = _log_int(rng, 33, 32768)
        per_token = 2 * S["kv_heads"] * S["hd"] * KV_BYTES[kv]
        hi = max(33, min(hi, int(3.0e9 / (per_token * batch))))
        lo = rng.randint(max(1, hi // 4), hi)
        layers = 4 if batch * hi * per_token < 6e7 else 1
        return _decode(shape, kv, batch, lo, hi, layers, rng.random() < 0.5, page)
    if kind == "prefill":
        batch = rng.choice((1, 1, 1, 2, 4))
        prompt = _log_int(rng, 40, 3000)
        start = rng.choice((0, 0, rng.randint(1, 6000)))
        chunk = rng.choice((128, 256, 512, 1024))
        if kv == "q4_0" and S["hd"] == 64:
            # no matrix-core kernel takes this cache: short prompts only
            batch, prompt, start = 1, min(prompt, 400), min(start, 400)
        while 4.0 * S["hd"] * S["heads"] * batch * prompt * (start + prompt / 2) > 2.5e11:
            batch, start = (batch // 2, start) if batch > 1 else (batch, start // 2)
        return _prefill(shape, kv, batch, start, prompt, min(chunk, prompt), rng.random() < 0.5, page)
    if kind == "matmul":
        dim = {"tinyllama": 2048, "llama8b": 4096, "llama70b": 8192}[shape]
        batch = _log_int(rng, 1, 512)
        if dim == 8192:
            batch = min(batch, 200)
        layers = 8 if batch <= 32 and dim < 8192 else 2
        return _matmul(rng.choice(sorted(WT)), dim, dim, batch, layers)
    return _get(shape, kv, _log_int(rng, 20, 16000), rng.random() < 0.5, page)


# ---- inputs ----------------------------------------------------------------

DEV = "cuda"


def _gen(seed, *tags):
    g = torch.Generator(device=DEV)
    s = seed & 0xFFFFFFFF
    for t in tags:
        s = (s * 1000003 + int(t) + 1) & 0x7FFFFFFFFFFF
    g.manual_seed(s)
    return g


def _kv_rows(seed, layer, seq, n, S):
    """K and V of n tokens of one sequence and layer: N(0, 1), K with a fixed
    spread over the dimensions (some are several times larger than others, as
    trained key projections have them)."""
    g = _gen(seed, 11, layer, seq)
    kd = S["kv_heads"] * S["hd"]
    spread = torch.exp(0.5 * torch.randn(kd, generator=_gen(seed, 12, layer), device=DEV))
    k = torch.randn(n, kd, generator=g, device=DEV) * spread
    v = torch.randn(n, kd, generator=g, device=DEV)
    return k, v


def _lens(case, seed):
    """Lengths spread evenly over [ctx_lo, ctx_hi], in an order of the seed."""
    b, lo, hi = case["batch"], case["ctx_lo"], case["ctx_hi"]
    lens = [hi if b == 1 else lo + (hi - lo) * i // (b - 1) for i in range(b)]
    order = np.random.default_rng(seed).permutation(b)
    return [lens[i] for i in order]


def _tables(lens, page, seed):
    """Block tables over a fragmented pool (pages handed out in random order):
    the int32 table, and the pool's page count."""
    need = [(n + page - 1) // page for n in lens]
    total = sum(need)
    pages = total + 8
    ids = np.random.default_rng(seed + 1).permutation(pages).astype(np.int32)
    bt = np.zeros((len(lens), max(need)), np.int32)
    o = 0
    for i, n in enumerate(need):
        bt[i, :n] = ids[o:o + n]
        o += n
    return bt, pages


def _dest(table_row, first, n, page):
    """Device (block ids, slots) of tokens first .. first + n - 1."""
    t = torch.arange(first, first + n, device=DEV)
    return table_row[t // page].to(torch.int32).contiguous(), (t % page).to(torch.int32).contiguous()


def _pool(case, layers, pages):
    S = SHAPES[case["shape"]]
    return gi.PagedKVCache(layers, S["kv_heads"], S["hd"], case["page"], pages, KV[case["kv"]])


def _scale(S):
    return float(gi.attn_scale(S["hd"]))


class _State:
    pass


def _prepare_decode(case, seed):
    S = SHAPES[case["shape"]]
    st = _State()
    lens = _lens(case, seed)
    bt, pages = _tables(lens, case["page"], seed)
    st.bt = torch.from_numpy(bt).to(DEV)
    st.lens = torch.tensor(lens, dtype=torch.int32, device=DEV)
    st.pool = _pool(case, case["layers"], pages)
    if case["rope"]:
        st.pool.SetRoPE(S["theta"], 0, max(lens) + 1)
    L, B, kd = case["layers"], case["batch"], S["kv_heads"] * S["hd"]
    st.q0 = torch.randn(L, B, S["heads"] * S["hd"], generator=_gen(seed, 1), device=DEV)
    st.q = st.q0.clone()
    st.k = torch.empty(L, B, kd, device=DEV)
    st.v = torch.empty(L, B, kd, device=DEV)
    st.out = torch.empty_like(st.q)
    for layer in range(L):
        for i, n in enumerate(lens):
            k, v = _kv_rows(seed, layer, i, n, S)
            st.k[layer, i], st.v[layer, i] = k[n - 1], v[n - 1]
            if n > 1:
                ids, slots = _dest(st.bt[i], 0, n - 1, case["page"])
                st.pool.Write(layer, ids, slots, k[:n - 1], v[:n - 1])
    # the calls of a token, arguments converted once (the buffers stay)
    method = "RoPEDecodeStep" if case["rope"] else "DecodeStep"
    st.calls = [st.pool.Prepare(method, st.out[la], st.q[la], st.k[la], st.v[la], la, st.bt, st.lens, S["heads"],
                                _scale(S), max_seq_len=max(lens)) for la in range(L)]
    st.pool.synchronize()
    return st


def _run_decode(st):
    if st.pool_rope:
        st.q.copy_(st.q0)  # the projection's output: RoPE turns q in place
    for call in st.calls:
        call()
    return [st.out]


def _chunks(case):
    n, c = case["prompt"], case["chunk"]
    return [(s, min(c, n - s)) for s in range(0, n, c)]


def _prepare_prefill(case, seed):
    S = SHAPES[case["shape"]]
    st = _State()
    B, page, start, total = case["batch"], case["page"], case["start"], case["start"] + case["prompt"]
    bt, pages = _tables([total] * B, page, seed)
    st.bt = torch.from_numpy(bt).to(DEV)
    st.pool = _pool(case, 1, pages)
    if case["rope"]:
        st.pool.SetRoPE(S["theta"], 0, total)
    st.heads, st.scale = S["heads"], _scale(S)
    ks, vs = zip(*[_kv_rows(seed, 0, i, total, S) for i in range(B)])
    for i in range(B):
        if start:
            ids, slots = _dest(st.bt[i], 0, start, page)
            st.pool.Write(0, ids, slots, ks[i][:start].contiguous(), vs[i][:start].contiguous())
    q = torch.randn(B, case["prompt"], S["heads"] * S["hd"], generator=_gen(seed, 1), device=DEV)
    st.chunks = []
    for s, n in _chunks(case):
        dest = [_dest(st.bt[i], start + s, n, page) for i in range(B)]
        c = _State()
        c.n = n
        c.ids = torch.cat([d[0] for d in dest])
        c.slots = torch.cat([d[1] for d in dest])
        c.k = torch.cat([k[start + s:start + s + n] for k in ks])
        c.v = torch.cat([v[start + s:start + s + n] for v in vs])
        c.q = q[:, s:s + n].contiguous().view(B * n, -1)
        c.q_out = torch.empty_like(c.q)
        c.out = torch.empty_like(c.q)
        c.pos = torch.arange(start + s, start + s + n, device=DEV, dtype=torch.int32).repeat(B)
        c.start = torch.full((B,), start + s, device=DEV, dtype=torch.int32)
        st.chunks.append(c)
    st.pool.synchronize()
    return st


def _run_prefill(st):
    for c in st.chunks:
        q = c.q
        if st.pool_rope:
            st.pool.RoPEWrite(0, c.pos, c.ids, c.slots, c.q, c.k, c.v, q_out=c.q_out)
            q = c.q_out
        else:
            st.pool.Write(0, c.ids, c.slots, c.k, c.v)
        st.pool.AttentionGQABatch(c.out, q, 0, st.bt, c.start, st.heads, st.scale, c.n)
    return [c.out for c in st.chunks]


def _weights(case, seed, layer):
    """One layer's weights: the GGUF bytes (host) and their float64 values
    (a function, made only when asked for)."""
    R, C = case["rows"], case["cols"]
    g = _gen(seed, 21, layer)
    w = torch.randn(R, C, generator=g, device=DEV) * 0.02
    t = case["wtype"]
    if t == "f32":
        return w.cpu().numpy(), lambda: w.double()
    if t == "f16":
        h = w.half()
        return h.cpu().numpy(), lambda: h.double()
    b = w.view(R, C // 32, 32)
    d = (b.abs().amax(2) / (127.0 if t == "q8_0" else 7.0)).half()
    dbytes = d.view(torch.uint8).view(R, C // 32, 2)
    x = b / d.float().unsqueeze(2)
    if t == "q8_0":
        q = x.round().clamp(-127, 127)
        raw = torch.cat([dbytes, q.to(torch.int8).view(torch.uint8)], 2)
    else:
        q = x.round().clamp(-8, 7)
        n = (q + 8).to(torch.uint8)
        raw = torch.cat([dbytes, n[..., :16] | (n[..., 16:] << 4)], 2)
    return (raw.reshape(-1).cpu().numpy(),
            lambda: (q.double() * d.double().unsqueeze(2)).view(R, C))


def _prepare_matmul(case, seed):
    st = _State()
    S = SHAPES["llama8b"]
    # the pool whose device and stream the products run on
    st.pool = gi.PagedKVCache(1, S["kv_heads"], S["hd"], 16, 4, gi.KV_F16)
    st.w, st.x, st.y = [], [], []
    for la in range(case["layers"]):
        raw, _ = _weights(case, seed, la)
        st.w.append(gi.Weights(st.pool, WT[case["wtype"]], case["rows"], case["cols"], raw))
        st.x.append(_activations(case, seed, la))
        st.y.append(torch.empty(case["batch"], case["rows"], device=DEV))
    st.pool.synchronize()
    return st


def _activations(case, seed, layer):
    return torch.randn(case["batch"], case["cols"], generator=_gen(seed, 22, layer), device=DEV)


def _run_matmul(st):
    for w, x, y in zip(st.w, st.x, st.y):
        w.MatMulBatch(y, x)
    return list(st.y)


def _prepare_get(case, seed):
    S = SHAPES[case["shape"]]
    st = _State()
    n = case["tokens"]
    bt, pages = _tables([n], case["page"], seed)
    st.bt = torch.from_numpy(bt[0]).to(DEV)
    st.pool = _pool(case, 1, pages)
    k, v = _kv_rows(seed, 0, 0, n, S)
    ids, slots = _dest(st.bt, 0, n, case["page"])
    st.pool.Write(0, ids, slots, k, v)
    st.tokens, st.widen = n, case["widen"]
    st.pool.synchronize()
    return st


def _run_get(st):
    return list(st.pool.Get(0, st.bt, st.tokens, widen=st.widen))


def prepare(case, seed):
    st = {"decode": _prepare_decode, "prefill": _prepare_prefill, "matmul": _prepare_matmul,
          "get": _prepare_get}[case["kind"]](case, seed)
    st.kind = case["kind"]
    st.pool_rope = case.get("rope", False)
    return st


def run(state):
    return {"decode": _run_decode, "prefill": _run_prefill, "matmul": _run_matmul,
            "get": _run_get}[state.kind](state)


# ---- what a pass cannot do without ------------------------------------------

def work(case):
    if case["kind"] == "matmul":
        R, C, B, L = case["rows"], case["cols"], case["batch"], case["layers"]
        per = {"f32": 4.0, "f16": 2.0, "q8_0": 34 / 32, "q4_0": 18 / 32}[case["wtype"]]
        return {"bytes": L * (R * C * per + 4 * B * (R + C)), "flops": L * 2 * B * R * C}
    S = SHAPES[case["shape"]]
    kd, qd, page = S["kv_heads"] * S["hd"], S["heads"] * S["hd"], case["page"]
    tok = 2 * kd * KV_BYTES[case["kv"]]  # stored bytes of a token
    if case["kind"] == "get":
        n = case["tokens"]
        return {"bytes": n * (tok + (2 * kd * 4 if case["widen"] else tok)) + 4 * -(-n // page), "flops": 0}
    if case["kind"] == "decode":
        lens = _lens(case, 0)
        n, B, L = sum(lens), case["batch"], case["layers"]
        # cached tokens, q and out, the new token in and stored, the table
        per_layer = (n - B) * tok + B * (8 * qd + 8 * kd + tok) + sum(4 * -(-x // page) for x in lens)
        return {"bytes": L * per_layer, "flops": L * 4 * qd * n}
    # prefill: the context is read once (whatever the chunks), q in, out out,
    # K / V in and stored
    B, n, start = case["batch"], case["prompt"], case["start"]
    pairs = sum(start + i + 1 for i in range(n))
    return {"bytes": B * (start * tok + n * (8 * qd + 8 * kd + tok) + 4 * -(-(start + n) // page)),
            "flops": B * 4 * qd * pairs}


# ---- tolerances ---------------------------------------------------------------

def tolerance(case):
    """Operands are exact (the cache and the weights are compared as stored)
    and every product and sum has float32 accuracy, so what is left is
    summation order, exp and the split of float32 operands: about four times
    the largest difference measured against float64."""
    if case["kind"] == "get":
        return "exact"
    return {"rel": 1e-5, "max": 1.6e-4}


# ---- the same in float64 --------------------------------------------------------

def _trunc_half(x):
    """float32 -> half, dropping mantissa bits (the cache's fp16 form)."""
    h = x.half()
    over = h.float().abs() > x.abs()
    return (h.view(torch.int16) - over.to(torch.int16)).view(torch.half)


def _quantised(kv, x):
    """The codes [n, blocks, 32] (float64) and block scales [n, blocks]
    (half) of rows x [n, kv_dim] in a q8_0 or q4_0 cache."""
    b = x.view(x.shape[0], -1, 32)
    q = 127.0 if kv == "q8_0" else 7.0
    d = _trunc_half((b.abs().amax(2).double() / q).float())
    inv = torch.where(d > 0, 1.0 / d.double(), torch.zeros((), dtype=torch.float64, device=x.device)).float()
    t = (b * inv.unsqueeze(2)).double()
    t = torch.sign(t) * torch.floor(t.abs() + 0.5)
    return (t.clamp(-128, 127) if kv == "q8_0" else t.clamp(-8, 7)), d


def _stored(kv, x):
    """The values rows x [n, kv_dim] have once stored in the cache, float64."""
    if kv == "f32":
        return x.double()
    if kv == "f16":
        return _trunc_half(x).double()
    t, d = _quantised(kv, x)
    return (t * d.double().unsqueeze(2)).view(x.shape)


def _stored_bytes(kv, x):
    """The bytes rows x [n, kv_dim] have in the host's cache layout."""
    if kv == "f32":
        return x.contiguous().view(torch.uint8)
    if kv == "f16":
        return _trunc_half(x).view(torch.uint8)
    t, d = _quantised(kv, x)
    dbytes = d.unsqueeze(2).view(torch.uint8)
    if kv == "q8_0":
        codes = t.to(torch.int8).view(torch.uint8)
    else:
        n = (t + 8).to(torch.uint8)
        codes = n[..., :16] | (n[..., 16:] << 4)
    return torch.cat([dbytes, codes], 2).view(x.shape[0], -1)


def _rope(x, pos, S):
    """x [n, heads * hd] turned at positions pos [n]: float32 products, each
    rounded, of cos and sin rounded from float64."""
    hd = S["hd"]
    half = hd // 2
    freq = 1.0 / S["theta"] ** (2.0 * torch.arange(half, device=x.device, dtype=torch.float64) / hd)
    ang = pos.double().unsqueeze(1) * freq
    c, s = ang.cos().float().unsqueeze(1), ang.sin().float().unsqueeze(1)
    y = x.view(x.shape[0], -1, hd)
    a, b = y[..., :half], y[..., half:]
    return torch.cat([a * c - b * s, a * s + b * c], 2).view(x.shape)


def _attend(q, K, V, S, first):
    """q [m, H * hd] at positions first .. first + m - 1 over K, V [n, kvh *
    hd] (float64, causal); [m, H * hd]."""
    H, kvh, hd = S["heads"], S["kv_heads"], S["hd"]
    m, n = q.shape[0], K.shape[0]
    G = H // kvh
    qh = q.double().view(m, kvh, G, hd).permute(1, 2, 0, 3).reshape(kvh, G * m, hd)
    kh = K.view(n, kvh, hd).permute(1, 2, 0).contiguous()
    s = torch.bmm(qh, kh).view(kvh, G, m, n) * _scale(S)
    if m > 1:
        t = torch.arange(n, device=q.device)
        p = torch.arange(first, first + m, device=q.device)
        s.masked_fill_(t.unsqueeze(0) > p.unsqueeze(1), float("-inf"))
    s = torch.softmax(s, -1).view(kvh, G * m, n)
    o = torch.bmm(s, V.view(n, kvh, hd).permute(1, 0, 2).contiguous())
    return o.view(kvh, G, m, hd).permute(2, 0, 1, 3).reshape(m, H * hd)


def exact(case, seed):
    if case["kind"] == "get":
        rows = _kv_rows(seed, 0, 0, case["tokens"], SHAPES[case["shape"]])
        form = _stored if case["widen"] else _stored_bytes
        return [form(case["kv"], x) for x in rows]
    if case["kind"] == "matmul":
        out = []
        for la in range(case["layers"]):
            w = _weights(case, seed, la)[1]()
            out.append(torch.mm(_activations(case, seed, la).double(), w.t().contiguous()))
        return out
    S = SHAPES[case["shape"]]
    if case["kind"] == "decode":
        lens = _lens(case, seed)
        q = torch.randn(case["layers"], case["batch"], S["heads"] * S["hd"], generator=_gen(seed, 1), device=DEV)
        out = torch.empty(q.shape, dtype=torch.float64, device=DEV)
        for la in range(case["layers"]):
            for i, n in enumerate(lens):
                k, v = _kv_rows(seed, la, i, n, S)
                qi = q[la, i:i + 1]
                if case["rope"]:
                    pos = torch.tensor([n - 1], device=DEV)
                    qi = _rope(qi, pos, S)
                    k[n - 1:] = _rope(k[n - 1:], pos, S)
                out[la, i] = _attend(qi, _stored(case["kv"], k), _stored(case["kv"], v), S, n - 1)[0]
        return [out]
    B, start = case["batch"], case["start"]
    q = torch.randn(B, case["prompt"], S["heads"] * S["hd"], generator=_gen(seed, 1), device=DEV)
    outs = [torch.empty(B, n, S["heads"] * S["hd"], dtype=torch.float64, device=DEV) for _, n in _chunks(case)]
    for i in range(B):
        k, v = _kv_rows(seed, 0, i, start + case["prompt"], S)
        pos = torch.arange(start, start + case["prompt"], device=DEV)
        qi = q[i]
        if case["rope"]:
            qi = _rope(qi, pos, S)
            k[start:] = _rope(k[start:], pos, S)
        K, V = _stored(case["kv"], k), _stored(case["kv"], v)
        for (s, n), o in zip(_chunks(case), outs):
            end = start + s + n
            o[i] = _attend(qi[s:s + n], K[:end], V[:end], S, start + s)
    return [o.view(-1, S["heads"] * S["hd"]) for o in outs]
