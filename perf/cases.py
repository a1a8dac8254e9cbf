"""Performance cases of the framework: the calls a program makes, over the sizes it makes them at.

Five kinds of case, each a dict of plain values:

  linear    one W4A8 product on device pointers (rai_w4a8_matmul_noalloc_dev where the
            activations fit its scratch, rai_w4a8_matmul_dev above), 1 token (decode),
            a few (verify batches) or many (prefill), group 32, 64 or 128
  fused     the one-token fused projections (rai_w4a8_fused_qkv_dev /
            rai_w4a8_fused_gate_up_dev)
  tied      the tied 8-bit lm_head (rai_tied_lm_head_dev)
  forward   a transformer block through RaiModel.forward_batch at a filled KV cache, with
            RaiModel.hidden_to_logits_batch where a program wants logits
  generate  a decoder's greedy loop (LookupDecoder.greedy_decode) from a prefilled
            prompt, then the logits after its last token
"""
import math

import numpy as np
import torch  # before rai_amd, so that both use one HIP runtime

import rai_amd

# Shapes of the benchmarked model families (hidden, heads, kv heads, head size, FFN, vocabulary).
TINYLLAMA = dict(hidden=2048, heads=32, kv_heads=4, head_dim=64, ffn=5632, vocab=32000, experts=0, topk=0)
MISTRAL = dict(hidden=4096, heads=32, kv_heads=8, head_dim=128, ffn=14336, vocab=32000, experts=0, topk=0)
OLMOE = dict(hidden=2048, heads=16, kv_heads=16, head_dim=128, ffn=1024, vocab=50304, experts=64, topk=8)


def _linear(rows, cols, tokens, group):
    return {"kind": "linear", "rows": rows, "cols": cols, "tokens": tokens, "group": group}


def _forward(shape, group, tokens, pos, logits, tied=False):
    return {"kind": "forward", **shape, "layers": 1, "group": group, "tokens": tokens, "pos": pos,
            "logits": logits, "tied": tied}


def listed():
    cases = {
        # The smallest call: TinyLlama's output projection for one decoded token.
        "matvec_2048x2048_g32": _linear(2048, 2048, 1, 32),
        # One decoded token through the MLP's first half, Mistral-7B shape.
        "gate_up_14336x4096_g32": {"kind": "fused", "rows": "14336,14336", "cols": 4096, "group": 32},
        # A lookup verify batch (8 drafts + 1) through the largest projection.
        "verify9_28672x4096_g32": _linear(28672, 4096, 9, 32),
        # The same batch at the reference's own group size, the long-row projection.
        "verify9_4096x14336_g128": _linear(4096, 14336, 9, 128),
        # A prefill chunk at group 128.
        "prefill512_14336x4096_g128": _linear(14336, 4096, 512, 128),
        # A prompt of odd length through a Llama-2-7B-like down projection.
        "prefill301_4096x11008_g32": _linear(4096, 11008, 301, 32),
        # Head of a model with tied 8-bit embeddings, one token.
        "tied_head_32000x2048": {"kind": "tied", "vocab": 32000, "hidden": 2048, "group": 64},
        # A short completion: the whole TinyLlama-shaped model, eight greedy tokens.
        "generate8_tinyllama": {"kind": "generate", **TINYLLAMA, "layers": 22, "group": 32, "prompt": 128,
                                "tokens": 8},
        # One token through a group-128 Mistral-shaped layer and head at 1000 positions.
        "decode_mistral_g128": _forward(MISTRAL, 128, 1, 1000, True),
        # A verify batch at a long context, with its nine rows of logits.
        "verify9_mistral_ctx4096": _forward(MISTRAL, 32, 9, 4096, True),
        # The last chunk of a 4096-token prompt.
        "prefill1024_mistral_ctx3072": _forward(MISTRAL, 32, 1024, 3072, False),
        # A prompt through a sparse layer (64 experts, 8 per token).
        "prefill512_olmoe": _forward(OLMOE, 32, 512, 0, False),
    }
    return [dict(c, name=n) for n, c in cases.items()]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _tokens(rng, most):
    """Decode, a verify batch, a short prompt or a prefill chunk."""
    lo, hi = rng.choice([(1, 1), (2, 17), (2, 64), (65, 512), (65, 512)])
    return min(most, _log(rng, lo, hi))


def draw(rng):
    kind = rng.choice(["linear"] * 9 + ["fused"] * 2 + ["tied"] * 2 + ["forward"] * 7)
    group = rng.choice([32, 32, 32, 64, 128, 128])
    if kind == "linear":
        while True:
            rows, cols = _log(rng, 256, 32768), group * max(1, _log(rng, 512, 14336) // group)
            tokens = _tokens(rng, 512)
            if rows * cols * tokens <= 14336 * 4096 * 512:
                return _linear(rows, cols, tokens, group)
    if kind == "fused":
        cols = group * max(1, _log(rng, 1024, 8192) // group)
        if rng.random() < 0.5:
            kv = 64 * rng.randint(4, 32)
            rows = [kv * rng.choice([1, 2, 4, 8]), kv, kv]
        else:
            rows = [_log(rng, 2048, 14336)] * 2
        return {"kind": "fused", "rows": ",".join(map(str, rows)), "cols": cols, "group": group}
    if kind == "tied":
        egs = rng.choice([32, 64, 64, 128])
        return {"kind": "tied", "vocab": _log(rng, 8192, 65536), "hidden": egs * max(4, _log(rng, 512, 4096) // egs),
                "group": egs}
    hd = rng.choice([64, 128])
    kv = rng.choice([1, 2, 4, 8])
    per = rng.choice([1, 2, 4, 8])
    while kv * per * hd < 512 or kv * per * hd > 4096:
        kv, per = rng.choice([1, 2, 4, 8]), rng.choice([1, 2, 4, 8])
    hidden = kv * per * hd
    experts = rng.choice([0, 0, 0, 8, 32])
    ffn = 256 * rng.randint(1, 4) if experts else 128 * rng.randint(hidden // 64, hidden // 32)
    shape = dict(hidden=hidden, heads=kv * per, kv_heads=kv, head_dim=hd, ffn=ffn, vocab=_log(rng, 4096, 50304),
                 experts=experts, topk=min(experts, rng.choice([2, 4, 8])))
    tokens = _tokens(rng, 512)
    pos = rng.choice([0, _log(rng, 16, 4096)])
    return _forward(shape, group, tokens, pos, tokens <= 64, rng.random() < 0.3)


# ----------------------------------------------------------------- inputs --

def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed) * 7919 + 17)


def _weights(g, rows, cols, group):
    """N(0, 0.02) weights, min/max round to nearest into 4 bits: nibbles [rows][cols / 2], params
    [rows][cols / group][scale, zero]."""
    w = torch.empty(rows, cols // group, group, device="cuda").normal_(0.0, 0.02, generator=g)
    lo, hi = w.amin(2), w.amax(2)
    scale = ((hi - lo) / 15).clamp_min(1e-7).half()
    zero = lo.half()
    q = ((w - zero.float()[..., None]) / scale.float()[..., None]).round_().clamp_(0, 15).to(torch.uint8)
    q = q.view(rows, cols)
    return (q[:, 0::2] | (q[:, 1::2] << 4)).contiguous(), torch.stack([scale, zero], 2).contiguous()


def _table(g, vocab, hidden, group):
    """An 8-bit embedding table of the same weights: codes [vocab][hidden], params
    [vocab][hidden / group][scale, zero]."""
    groups = -(-hidden // group)
    w = torch.empty(vocab, groups, group, device="cuda").normal_(0.0, 0.02, generator=g)
    lo, hi = w.amin(2), w.amax(2)
    scale = ((hi - lo) / 255).clamp_min(1e-7).half()
    zero = lo.half()
    q = ((w - zero.float()[..., None]) / scale.float()[..., None]).round_().clamp_(0, 255).to(torch.uint8)
    return q.view(vocab, groups * group)[:, :hidden].contiguous(), torch.stack([scale, zero], 2).contiguous()


def _acts(g, tokens, cols):
    return torch.empty(tokens, cols, device="cuda").normal_(0.0, 1.0, generator=g)


def _projections(c):
    """(rows, cols) of a layer's seven linears in file order."""
    h, f, qd, kvd = c["hidden"], c["ffn"], c["heads"] * c["head_dim"], c["kv_heads"] * c["head_dim"]
    return [(qd, h), (kvd, h), (kvd, h), (h, qd), (f, h), (f, h), (h, f)]


def _embed_group(c):
    return 64 if c["hidden"] % 64 == 0 else 32


def _max_context(c):
    return 512 if c["kind"] == "generate" else max(512, c["pos"] + c["tokens"])


def _model_tensors(c, g):
    """The model's weights on the GPU: (embedding, layers, head); a layer is its linears (with the
    experts past the first after them) and its router."""
    emb = _table(g, c["vocab"], c["hidden"], _embed_group(c))
    layers = []
    for _ in range(c["layers"]):
        dims = _projections(c)
        lin = [_weights(g, r, k, c["group"]) for r, k in dims]
        router = None
        if c["experts"]:
            router = torch.empty(c["experts"], c["hidden"], device="cuda").normal_(0.0, 0.02, generator=g)
            for _ in range(c["experts"] - 1):
                lin += [_weights(g, r, k, c["group"]) for r, k in dims[4:]]
        layers.append((lin, router))
    head = None if c.get("tied") else _weights(g, c["vocab"], c["hidden"], c["group"])
    return emb, layers, head


def _bytes(t):
    return t.cpu().contiguous().numpy().reshape(-1).view(np.uint8)


def _image(c, tensors):
    """The .raimodel file of these weights (norm vectors of ones), as bytes."""
    emb, layers, head = tensors
    ones = np.ones(c["hidden"], np.float32).view(np.uint8)

    def linear(w):
        nib, par = w
        dims = np.array([nib.shape[0], nib.shape[1] * 2], np.uint32).view(np.uint8)
        return [dims, _bytes(par), _bytes(nib)]

    sections = [[_bytes(emb[1]), _bytes(emb[0])]]
    for lin, router in layers:
        s = [b for w in lin[:7] for b in linear(w)]
        if router is not None:
            s.append(_bytes(router))
            s += [b for w in lin[7:] for b in linear(w)]
        sections.append(s + [ones, ones])
    sections.append([ones])
    if head is not None:
        sections.append(linear(head))
    v2 = c["experts"] > 0
    header = np.zeros(128 if v2 else 64, np.uint8)
    header[:4] = np.frombuffer(b"RAIM", np.uint8)
    header[4:40] = np.array([2 if v2 else 1, c["hidden"], c["layers"], c["heads"], c["kv_heads"], c["head_dim"],
                             c["ffn"], c["vocab"], _max_context(c)], np.uint32).view(np.uint8)
    header[40:48] = np.array([10000.0, 1e-5], np.float32).view(np.uint8)
    header[48:52] = [4, c["group"], 8, _embed_group(c)]
    header[52:56] = np.array([len(sections)], np.uint32).view(np.uint8)
    if v2:
        header[84:88] = np.array([1.0], np.float32).view(np.uint8)
        header[105:107] = np.array([c["experts"]], np.uint16).view(np.uint8)
        header[107] = c["topk"]
    table, off = [], len(header) + 16 * len(sections)
    for s in sections:
        n = sum(b.size for b in s)
        table += [off, n]
        off += n
    return np.concatenate([header, np.array(table, np.uint64).view(np.uint8)] + [b for s in sections for b in s])


def _prompt(c, seed):
    """prompt + 1 token ids: the prefilled ones and the first to decode from."""
    return np.random.default_rng(seed).integers(0, c["vocab"], c["prompt"] + 1).astype(np.uint32)


def _forward_inputs(c, g):
    """The batch's hidden states and the cached K, V rows [layer][kv_head][pos][head_dim]."""
    x = _acts(g, c["tokens"], c["hidden"])
    kv = torch.empty(2, c["layers"], c["kv_heads"], c["pos"], c["head_dim"], device="cuda").normal_(generator=g)
    return x, kv


def prepare(case, seed):
    c, g = case, _gen(seed)
    if c["kind"] == "linear":
        nib, par = _weights(g, c["rows"], c["cols"], c["group"])
        x = _acts(g, c["tokens"], c["cols"])
        out = torch.zeros(c["tokens"], c["rows"], device="cuda")
        # The allocation-free call takes up to 2^20 activations (token counts padded to its tiles).
        fits = -(-c["tokens"] // 32) * 32 * c["cols"] <= 1 << 20 or c["tokens"] * c["cols"] * 4 <= 1 << 20
        lib = rai_amd.lib()
        fn = lib.rai_w4a8_matmul_noalloc_dev if fits else lib.rai_w4a8_matmul_dev
        return {"kind": "linear", "fn": fn, "nib": nib, "par": par, "x": x, "out": out, "case": c}
    if c["kind"] == "fused":
        rows = [int(r) for r in c["rows"].split(",")]
        w = [_weights(g, r, c["cols"], c["group"]) for r in rows]
        x = _acts(g, 1, c["cols"])
        outs = [torch.zeros(r, device="cuda") for r in rows]
        lins = [rai_amd.QLinear(n.data_ptr(), p.data_ptr(), r, c["cols"], c["group"]) for (n, p), r in zip(w, rows)]
        return {"kind": "fused", "w": w, "x": x, "outs": outs, "lins": lins}
    if c["kind"] == "tied":
        codes, par = _table(g, c["vocab"], c["hidden"], c["group"])
        x = _acts(g, 1, c["hidden"])
        return {"kind": "tied", "codes": codes, "par": par, "x": x,
                "out": torch.zeros(c["vocab"], device="cuda"), "case": c}
    # Groups of the longest rows, where they pass the loader's default bound of 128.
    groups = max(128, -(-max(k for _, k in _projections(c)) // c["group"]))
    model = rai_amd.RaiModel.from_bytes(_image(c, _model_tensors(c, g)), groups)
    if c["kind"] == "generate":
        dec = rai_amd.LookupDecoder(model, _max_context(c))
        ctx = _prompt(c, seed)
        pos = dec.prefill(ctx)
        return {"kind": "generate", "model": model, "dec": dec, "ctx": ctx, "pos": pos, "case": c}
    x, kv_rows = _forward_inputs(c, g)
    kv = model.create_kv_cache(_max_context(c))
    if c["pos"]:
        rows = kv_rows.cpu().numpy()
        for layer in range(c["layers"]):
            for which in (0, 1):
                kv.import_rows(layer, which, rows[which, layer])
    return {"kind": "forward", "model": model, "kv": kv, "x": x.cpu().numpy(),
            "positions": np.arange(c["pos"], c["pos"] + c["tokens"]), "case": c}


# -------------------------------------------------------------------- run --

def _check(rc):
    if rc:
        raise RuntimeError(rai_amd.lib().rai_last_error().decode())


def run(state):
    kind = state["kind"]
    if kind in ("linear", "fused", "tied"):
        lib, stream = rai_amd.lib(), torch.cuda.current_stream().cuda_stream
        if kind == "linear":
            c = state["case"]
            _check(state["fn"](state["out"].data_ptr(), state["nib"].data_ptr(), state["par"].data_ptr(),
                               state["x"].data_ptr(), c["rows"], c["cols"], c["tokens"], c["group"], stream))
            return state["out"]
        if kind == "fused":
            fn = lib.rai_w4a8_fused_qkv_dev if len(state["outs"]) == 3 else lib.rai_w4a8_fused_gate_up_dev
            _check(fn(*[o.data_ptr() for o in state["outs"]], *state["lins"], state["x"].data_ptr(), stream))
            return state["outs"]
        c = state["case"]
        _check(lib.rai_tied_lm_head_dev(state["out"].data_ptr(), state["x"].data_ptr(), state["codes"].data_ptr(),
                                        state["par"].data_ptr(), c["vocab"], c["hidden"], c["group"], stream))
        return state["out"]
    c, model = state["case"], state["model"]
    if kind == "generate":
        dec, pos = state["dec"], state["pos"]
        dec.kv_cache.truncate(pos)
        toks = dec.greedy_decode(state["ctx"], pos, c["tokens"])
        h = model.forward_from_hidden(model.embed_token(toks[-1]), pos + c["tokens"], dec.kv_cache)
        return {"tokens": np.array(toks), "logits": model.hidden_to_logits(h)}
    kv = state["kv"]
    kv.truncate(c["pos"])  # the call may be repeated: the batch's own rows are dropped
    h = model.forward_batch(state["x"], state["positions"], kv)
    out = {"hidden": h}
    if c["logits"]:
        out["logits"] = model.hidden_to_logits_batch(h, c["tokens"])
    return out


# ------------------------------------------------------------------- work --

def _w4_bytes(rows, cols, group):
    return rows * cols // 2 + 4 * rows * -(-cols // group)


def work(case):
    c = case
    if c["kind"] == "linear":
        r, k, m = c["rows"], c["cols"], c["tokens"]
        return {"bytes": _w4_bytes(r, k, c["group"]) + 4 * m * (r + k), "flops": 2 * r * k * m}
    if c["kind"] == "fused":
        rows, k = sum(int(r) for r in c["rows"].split(",")), c["cols"]
        return {"bytes": _w4_bytes(rows, k, c["group"]) + 4 * (rows + k), "flops": 2 * rows * k}
    if c["kind"] == "tied":
        v, h = c["vocab"], c["hidden"]
        return {"bytes": v * (h + 4 * -(-h // c["group"])) + 4 * (v + h), "flops": 2 * v * h}
    h, hd, nkv, nh, m = c["hidden"], c["head_dim"], c["kv_heads"], c["heads"], c["tokens"]
    dims = _projections(c)
    pos = c["prompt"] if c["kind"] == "generate" else c["pos"]

    def layer_pass(m, pos):
        # Weights of the dense projections once; of the experts, those that m tokens reach; the keys and
        # values up to each token once per pass, the new rows written once.
        by = sum(_w4_bytes(r, k, c["group"]) for r, k in dims[:4])
        fl = 2 * m * sum(r * k for r, k in dims[:4]) + 4 * nh * hd * sum(range(pos + 1, pos + m + 1))
        mlp_b, mlp_f = sum(_w4_bytes(r, k, c["group"]) for r, k in dims[4:]), 2 * sum(r * k for r, k in dims[4:])
        if c["experts"]:
            by += min(c["experts"], m * c["topk"]) * mlp_b + 4 * c["experts"] * h
            fl += m * (c["topk"] * mlp_f + 2 * c["experts"] * h)
        else:
            by, fl = by + mlp_b, fl + m * mlp_f
        return by + 8 * nkv * hd * (pos + m), fl

    if c["kind"] == "generate":
        by = fl = 0
        for i in range(m + 1):
            b, f = layer_pass(1, pos + i)
            by += c["layers"] * b + _w4_bytes(c["vocab"], h, c["group"])
            fl += c["layers"] * f + 2 * c["vocab"] * h
        return {"bytes": by + 4 * c["vocab"], "flops": fl}
    b, f = layer_pass(m, pos)
    by, fl = c["layers"] * b + 8 * m * h, c["layers"] * f
    if c["logits"]:
        v = c["vocab"]
        by += (v * (h + 4 * -(-h // _embed_group(c))) if c["tied"] else _w4_bytes(v, h, c["group"])) + 4 * m * v
        fl += 2 * m * v * h
    return {"bytes": by, "flops": fl}


def tolerance(case):
    # A single product: f32 sums of exact integer products (3e-7 to 1.1e-6 against 64 bits).  Blocks: a
    # last-bit difference moves an int8 activation across a rounding boundary here and there, and each of
    # the block's four quantizations takes the root of what came before it (1e-7 becomes 1e-3 to 2e-2
    # against 64 bits after one layer, where it stays: the step of the int8 grid itself).
    if case["kind"] in ("linear", "fused", "tied"):
        return {"rel": 4e-6}
    return {"rel": 3e-2, "max": 0.3, "differ": 0.0}


# ------------------------------------------------------------------ exact --

def _quant(x, group, top):
    """The path's activation rounding (part of what it computes): codes per group of f32 values, as f64,
    the scales and the sums of the raw values."""
    m, k = x.shape
    groups = -(-k // group)
    v = x.float()
    if groups * group != k:
        v = torch.nn.functional.pad(v, (0, groups * group - k))
    v = v.view(m, groups, group)
    a = v.abs().amax(2)
    s = torch.where(a > 1e-10, (a.double() / top).float(), torch.ones_like(a))
    q = (v * (1.0 / s.double()).float()[..., None]).round_().clamp_(-top - 1 if top == 127 else -top, top)
    sums = torch.nn.functional.pad(x, (0, groups * group - k)).double().view(m, groups, group).sum(2)
    return q.double(), s.double(), sums


def _product(x, codes, par, group, top):
    """x [m][k] against codes [rows][k] (f64 of integers) and params, in 64 bits."""
    q, s, sums = _quant(x, group, top)
    m, groups = s.shape
    a = (q * s[..., None]).view(m, -1)
    par = par.double()
    out = torch.empty(m, codes.shape[0], dtype=torch.float64, device=x.device)
    for r in range(0, codes.shape[0], 4096):
        w = codes[r:r + 4096].double()
        w = torch.nn.functional.pad(w, (0, groups * group - w.shape[1])).view(-1, groups, group)
        w = (w * par[r:r + 4096, :, :1]).view(-1, groups * group)
        out[:, r:r + 4096] = a @ w.t() + sums @ par[r:r + 4096, :, 1].t()
    return out


def _lin64(x, w, group):
    nib, par = w
    codes = torch.stack([nib & 15, nib >> 4], 2).view(nib.shape[0], -1)
    return _product(x, codes, par, group, 127)


def _norm64(x):
    return x / (x.square().mean(1, keepdim=True) + 1e-5).sqrt()


def _exp_body(d):
    """The path's exponential (Schraudolph 1999, part of what it computes), on f32 values."""
    v = (d.float() * 12102203.0 + 1064866816.0).clamp(0.0, 2139095040.0)
    return v.round().to(torch.int32).view(torch.float32).double()


def _rope64(x, pos, heads, hd):
    m, half = x.shape[0], hd // 2
    inv = np.float32(1.0) / np.power(np.float32(10000.0), np.arange(half, dtype=np.float32) * np.float32(2.0) /
                                     np.float32(hd))
    ang = (np.arange(pos, pos + m, dtype=np.float32)[:, None] * inv[None, :].astype(np.float32)).astype(np.float64)
    co, si = (torch.from_numpy(f(ang)).to(x.device)[:, None] for f in (np.cos, np.sin))
    v = x.view(m, heads, 2, half)
    a, b = v[:, :, 0], v[:, :, 1]
    return torch.stack([a * co - b * si, b * co + a * si], 2).view(m, heads, hd)


def _attention64(q, k, v, pos):
    """q [m][nh][hd] over k, v [nkv][pos + m][hd]: causal."""
    m, nh, hd = q.shape
    nkv, n = k.shape[0], k.shape[1]
    out = torch.empty(m, nh, hd, dtype=torch.float64, device=q.device)
    length = torch.arange(pos + 1, pos + m + 1, device=q.device)[:, None]
    at = torch.arange(n, device=q.device)[None]
    for h in range(nh):
        kh = h // (nh // nkv)
        s = (q[:, h] @ k[kh].t()) / math.sqrt(hd)
        s = s.masked_fill(at >= length, -math.inf)
        d = s - s.amax(1, keepdim=True)
        e = torch.where(at < length // 8 * 8, _exp_body(d.clamp_min(-200.0)), d.exp())
        e = e.masked_fill(at >= length, 0.0)
        out[:, h] = (e / e.sum(1, keepdim=True)) @ v[kh]
    return out.view(m, nh * hd)


def _mlp64(x, gate, up, down, group):
    a, b = _lin64(x, gate, group), _lin64(x, up, group)
    return _lin64(a / (1.0 + _exp_body(-a)) * b, down, group)


def exact(case, seed):
    c, g = case, _gen(seed)
    if c["kind"] == "linear":
        w = _weights(g, c["rows"], c["cols"], c["group"])
        return _lin64(_acts(g, c["tokens"], c["cols"]), w, c["group"])
    if c["kind"] == "fused":
        w = [_weights(g, int(r), c["cols"], c["group"]) for r in c["rows"].split(",")]
        x = _acts(g, 1, c["cols"])
        return [_lin64(x, p, c["group"])[0] for p in w]
    if c["kind"] == "tied":
        codes, par = _table(g, c["vocab"], c["hidden"], c["group"])
        return _product(_acts(g, 1, c["hidden"]), codes, par, c["group"], 63)[0]
    if c["kind"] == "generate":
        return None  # each token is the argmax of a model that ran on the ones before it: no value in other rounding
    emb, layers, head = _model_tensors(c, g)
    x, kv = _forward_inputs(c, g)
    x, kv = x.double(), kv.double()
    m, pos, nh, nkv, hd, gs = c["tokens"], c["pos"], c["heads"], c["kv_heads"], c["head_dim"], c["group"]
    for li, (lin, router) in enumerate(layers):
        n = _norm64(x)
        q = _rope64(_lin64(n, lin[0], gs), pos, nh, hd)
        k = _rope64(_lin64(n, lin[1], gs), pos, nkv, hd)
        v = _lin64(n, lin[2], gs).view(m, nkv, hd)
        k = torch.cat([kv[0, li], k.transpose(0, 1)], 1)
        v = torch.cat([kv[1, li], v.transpose(0, 1)], 1)
        x = x + _lin64(_attention64(q, k, v, pos), lin[3], gs)
        n = _norm64(x)
        if router is None:
            x = x + _mlp64(n, lin[4], lin[5], lin[6], gs)
            continue
        p = torch.softmax(n @ router.double().t(), 1)
        top, pick = p.topk(c["topk"], 1)
        add = torch.zeros_like(x)
        for e in range(c["experts"]):
            t, slot = (pick == e).nonzero(as_tuple=True)
            if t.numel():
                add[t] += top[t, slot][:, None] * _mlp64(n[t], *lin[4 + 3 * e:7 + 3 * e], gs)
        x = x + add
    out = {"hidden": x}
    if c["logits"]:
        n = _norm64(x)
        out["logits"] = (_product(n, emb[0], emb[1], _embed_group(c), 63) if c["tied"] else _lin64(n, head, gs))
    return out
