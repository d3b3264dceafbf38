"""Performance cases of the paged attention path, through its public entry points.

A case is a dict of plain values; ``kind`` names the entry point:

* ``step``: one decode step on bound buffers (``PreparedDecodeStep``:
  attention over every request's context, then the append of its new token),
  what a serving loop or a captured decode graph runs per layer;
* ``op``: the same work through the eager operators with their default
  value checks (``append_kv_hip`` + ``paged_decode_attention_hip_grouped``),
  the way a caller of the reference's operators uses them;
* ``prefill``: causal attention of a prompt chunk per request
  (``PreparedPagedPrefill``, the layer loop of a batched prefill);
* ``rope``: rotary embedding of a prefill batch's q and k fused with the
  append of its rows into the cache (``rope_append_kv_hip``);
* ``llama``: a whole run of a Llama model, batched prefill and greedy decode
  (``LlamaPagedDecodeRunner``).
"""

from __future__ import annotations

import math

import torch

DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}
DEVICE = "cuda"


def listed():
    return [
        # The smallest call: one request answered in a chat, a GQA layer of a
        # 7-8 B model.
        _decode("step_gqa_b1", "step", 1, 32, 8, 128, "bf16", 1000, 1000),
        # The eager operators at the size of the reference's smoke benchmark
        # (4 requests x 512 tokens, fp32, head_dim 64), values checked.
        _decode("op_gqa_fp32", "op", 4, 32, 8, 64, "fp32", 512, 512),
        # The eager operators at the reference's published sweep shape.
        _decode("op_gqa_fp16", "op", 16, 32, 8, 64, "fp16", 2048, 2048),
        # A multi-head layer: short contexts, every query head its own K/V.
        _decode("step_mha_fp16", "step", 16, 32, 32, 128, "fp16", 512, 512),
        # A multi-query layer: one K/V head for 32 query heads, ragged.
        _decode("step_mqa_bf16", "step", 64, 32, 1, 128, "bf16", 1024, 4096),
        # The default benchmark: long-context serving of a GQA model.
        _decode("step_gqa_bf16", "step", 32, 32, 8, 128, "bf16", 4096, 8192),
        # The same traffic over the FP8 cache.
        _decode("step_gqa_fp8", "step", 32, 32, 8, 128, "bf16", 4096, 8192, cache="fp8"),
        # A batch of long prompts, the largest case.
        _prefill("prefill_long_bf16", 8, 32, 8, 128, "bf16", 0, 0, 4096, 4096),
        # A batch of short prompts, as the Llama runner prefills them.
        _prefill("prefill_short_bf16", 8, 16, 4, 128, "bf16", 0, 0, 512, 512),
        # Ragged later chunks of long prompts over the FP8 cache.
        _prefill("prefill_chunk_fp8", 4, 32, 8, 128, "bf16", 1024, 3072, 517, 1024, cache="fp8"),
        # A full-precision check run: ragged prompts in fp32.
        _prefill("prefill_fp32", 4, 32, 8, 64, "fp32", 0, 0, 257, 512),
        # The tiny Llama (8 layers, 16/4 heads of 128): 16 prompts, 16 new
        # tokens each.
        {"name": "llama_bf16", "kind": "llama", "batch": 16, "lo": 384, "hi": 512, "new": 16, "layers": 8,
         "hidden": 2048, "inter": 5632, "heads": 16, "kv_heads": 4, "head_dim": 128, "vocab": 32000,
         "dtype": "bf16", "cache": "same", "block": 16, "budget": 4096},
    ]


def _decode(name, kind, batch, heads, kv_heads, head_dim, dtype, lo, hi, cache="same", block=16, index="i32"):
    case = {"kind": kind, "batch": batch, "heads": heads, "kv_heads": kv_heads, "head_dim": head_dim, "dtype": dtype,
            "lo": lo, "hi": hi, "cache": cache, "block": block, "index": index}
    return {"name": name, **case} if name else case


def _prefill(name, batch, heads, kv_heads, head_dim, dtype, start_lo, start_hi, lo, hi, cache="same", block=16):
    case = {"kind": "prefill", "batch": batch, "heads": heads, "kv_heads": kv_heads, "head_dim": head_dim,
            "dtype": dtype, "start_lo": start_lo, "start_hi": start_hi, "lo": lo, "hi": hi, "cache": cache,
            "block": block}
    return {"name": name, **case} if name else case


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["step", "step", "step", "op", "op", "prefill", "prefill", "prefill", "rope", "llama"])
    if kind == "llama":
        heads = rng.choice([8, 16])
        return {"kind": "llama", "batch": _log(rng, 1, 16), "lo": _log(rng, 16, 128), "hi": _log(rng, 129, 512),
                "new": rng.randint(2, 16), "layers": rng.randint(2, 8), "hidden": 128 * heads,
                "inter": 352 * heads, "heads": heads, "kv_heads": rng.choice([2, 4, 8]), "head_dim": 128,
                "vocab": 32000, "dtype": "bf16", "cache": rng.choice(["same", "same", "fp8"]), "block": 16,
                "budget": rng.choice([2048, 4096])}
    heads, kv_heads = rng.choice([(32, 32), (32, 8), (32, 8), (32, 4), (16, 4), (32, 1), (8, 2), (28, 4)])
    if kind == "rope":
        return {"kind": "rope", "tokens": _log(rng, 1, 8192), "heads": heads, "kv_heads": kv_heads,
                "head_dim": rng.choice([64, 128, 128]), "dtype": rng.choice(["bf16", "fp16"]),
                "cache": rng.choice(["same", "fp8"]), "block": 16}
    dtype = rng.choice(["bf16", "bf16", "bf16", "fp16", "fp16", "fp32"])
    head_dim = rng.choice([64, 64, 96, 128, 128, 128])
    block = rng.choice([16, 16, 16, 32])
    fp8 = dtype == "bf16" and rng.random() < 0.3
    cache = "fp8" if fp8 else "same"
    if kind == "prefill":
        batch = _log(rng, 1, 16)
        # at most the pairs of the largest listed case; an eighth of a
        # short-prompt batch in fp32
        most = 8 * 4096 if dtype != "fp32" else 2048
        hi = max(17, min(4096 if dtype != "fp32" else 1024, _log(rng, 33, 4096), most // batch))
        lo = rng.randint(max(1, hi // 2), hi)
        start_hi = 0 if dtype == "fp32" or rng.random() < 0.5 else rng.randint(1, max(1, min(3072, 4096 - hi)))
        return _prefill(None, batch, heads, kv_heads, head_dim, dtype, start_hi // 3, start_hi, lo, hi, cache, block)
    # decode: at most the K/V bytes of the default benchmark
    batch = _log(rng, 1, 64)
    row = kv_heads * head_dim * (4 if dtype == "fp32" else 2) * 2
    hi = max(32, min(8192, _log(rng, 100, 8192), 800_000_000 // (row * batch)))
    lo = rng.randint(max(1, hi // 3), hi)
    if kind == "op":
        # callers of the eager operators also come with other row widths,
        # block sizes and 64-bit metadata
        head_dim = rng.choice([head_dim, head_dim, 32])
        block = rng.choice([block, block, 8]) if not fp8 else block
        return _decode(None, "op", batch, heads, kv_heads, head_dim, dtype, lo, hi, cache, block,
                       rng.choice(["i32", "i64"]))
    return _decode(None, "step", batch, heads, kv_heads, head_dim, dtype, lo, hi, cache, block)


# ------------------------------------------------------------------ inputs
def _quantize(rows):
    """E4M3 codes and one power-of-two fp32 scale per row of ``rows``
    [..., D]: the smallest 2^k with amax / 2^k <= 448, 1 for a zero row."""
    x = rows.float()
    amax = x.abs().amax(-1, keepdim=True)
    m, e = torch.frexp(amax / 448.0)  # m in [0.5, 1): a power of two has m = 0.5
    scale = torch.ldexp(torch.ones_like(amax), torch.where(m == 0.5, e - 1, e).clamp_min(-126))
    scale = torch.where(amax == 0, torch.ones_like(scale), scale)
    return (x / scale).to(torch.float8_e4m3fn), scale.squeeze(-1)


def _sizes(case, seed):
    """Context lengths (decode) or (starts, spans) (prefill): which request
    is how long depends on the seed, the work of a case does not."""
    gen = torch.Generator().manual_seed(seed)

    def spread(lo, hi):
        n = case["batch"]
        even = [lo + (hi - lo) * (2 * i + 1) // (2 * n) for i in range(n)] if n > 1 else [hi]
        return [even[i] for i in torch.randperm(n, generator=gen).tolist()]

    if case["kind"] == "prefill":
        return spread(case["start_lo"], case["start_hi"]), spread(case["lo"], case["hi"])
    return spread(case["lo"], case["hi"])


def _fill(shape, seed, dtype):
    gen = torch.Generator(device=DEVICE).manual_seed(seed)
    return torch.empty(shape, dtype=dtype, device=DEVICE).normal_(0.0, 1.0, generator=gen)


def _inputs(case, seed):
    """Raw inputs on the GPU: the pool's K/V rows (or FP8 codes and scales),
    block tables, lengths, queries and new rows. Blocks come from a
    permuted pool, as a long-running server hands them out; the block that
    takes a request's new token is its newest, from the pool's end."""
    dtype, bs, batch = DTYPES[case["dtype"]], case["block"], case["batch"]
    hkv, d = case["kv_heads"], case["head_dim"]
    gen = torch.Generator().manual_seed(seed + 1)
    sizes = _sizes(case, seed)
    if case["kind"] == "prefill":
        starts, spans = sizes
        ends = [s + n for s, n in zip(starts, spans)]
        need = [-(-n // bs) for n in ends]
        pool = sum(need) + 8
        perm = torch.randperm(pool, generator=gen).tolist()
    else:
        ends = sizes
        need = [n // bs + 1 for n in ends]
        pool = sum(need) + 8
        perm = torch.randperm(pool - batch, generator=gen).tolist()
    tables, used = [], 0
    for b, n in enumerate(need):
        own = n if case["kind"] == "prefill" else n - 1
        tables.append(perm[used:used + own] + ([] if own == n else [pool - batch + b]))
        used += own
    width = max(need)
    raw = {"pool": pool, "ends": ends, "need": need,
           "tables": torch.tensor([t + [0] * (width - len(t)) for t in tables], dtype=torch.int32, device=DEVICE)}
    shape = (pool, bs, hkv, d)
    for i, name in enumerate(("k", "v")):
        x = _fill(shape, 4 * seed + i, dtype)
        if case["cache"] == "fp8":
            raw[name], raw[name + "_scale"] = _quantize(x)
        else:
            raw[name] = x
    if case["kind"] == "prefill":
        raw["starts"] = starts
        raw["q"] = _fill((batch, case["heads"], max(spans), d), 4 * seed + 2, dtype)
        return raw
    raw["q"] = _fill((batch, case["heads"], d), 4 * seed + 2, dtype)
    raw["new_k"], raw["new_v"] = _fill((2, batch, hkv, d), 4 * seed + 3, dtype)
    raw["lens"] = torch.tensor(ends, dtype=torch.int32, device=DEVICE)
    raw["slots"] = torch.tensor([t[n // bs] * bs + n % bs for t, n in zip(tables, ends)], dtype=torch.int32,
                                device=DEVICE)
    return raw


def _cache(case, raw):
    from inferkernellab_amd import PagedKVCache

    dtype = DTYPES[case["dtype"]]
    fp8 = case["cache"] == "fp8"
    cache = PagedKVCache(raw["pool"], case["block"], case["kv_heads"], case["head_dim"],
                         dtype=torch.float8_e4m3fn if fp8 else dtype, act_dtype=dtype if fp8 else None, device=DEVICE)
    for name in ("k", "v"):
        getattr(cache, name)[0].copy_(raw[name])
        if fp8:
            getattr(cache, name + "_scale")[0].copy_(raw[name + "_scale"].transpose(1, 2))
    return cache


def _parts(out, raw):
    """A prefill's output whole, as views of its parts: each request's rows
    (shortest chunk first), and the rows that pad it to the longest chunk (a
    row of V, far larger than an attention's mean over many)."""
    spans = sorted((e - s, b) for b, (s, e) in enumerate(zip(raw["starts"], raw["ends"])))
    return {"rows": [out[b, :, :n] for n, b in spans], "padding": [out[b, :, n:] for n, b in spans]}


def _blocks(cache, n):
    """The last n blocks of the cache: what a decode step updates."""
    out = {}
    for name in ("k", "v"):
        rows = getattr(cache, name)[0, -n:]
        if cache.fp8:
            out[name] = rows.view(torch.uint8)
            out[name + "_scale"] = getattr(cache, name + "_scale")[0, -n:]
        else:
            out[name] = rows
    return out


def _rope_inputs(case, seed):
    t, dtype, bs = case["tokens"], DTYPES[case["dtype"]], case["block"]
    h, hkv, d = case["heads"], case["kv_heads"], case["head_dim"]
    pool = -(-t // bs)
    gen = torch.Generator().manual_seed(seed)
    perm = torch.randperm(pool, generator=gen)
    at = torch.arange(t)
    slots = (perm[at // bs] * bs + at % bs).to(torch.int32).to(DEVICE)
    inv = 1.0 / (10000.0 ** (torch.arange(0, d, 2, dtype=torch.float32) / d))
    angles = torch.arange(t, dtype=torch.float32).unsqueeze(-1) * inv
    angles = torch.cat((angles, angles), dim=-1).to(DEVICE)
    return {"pool": pool, "slots": slots, "cos": angles.cos().to(dtype), "sin": angles.sin().to(dtype),
            "q": _fill((t, h, d), 4 * seed, dtype), "key": _fill((t, hkv, d), 4 * seed + 1, dtype),
            "value": _fill((t, hkv, d), 4 * seed + 2, dtype)}


def _llama_weights(case, seed):
    """Weights of a Llama whose next token is decided with the margin a
    trained model shows: embeddings ~ N(0, 1), and each output row a scaled
    embedding row of the token it follows."""
    dtype = DTYPES[case["dtype"]]
    hid, inter, d = case["hidden"], case["inter"], case["head_dim"]
    sizes = {"self_attn.q_proj": (case["heads"] * d, hid), "self_attn.k_proj": (case["kv_heads"] * d, hid),
             "self_attn.v_proj": (case["kv_heads"] * d, hid), "self_attn.o_proj": (hid, case["heads"] * d),
             "mlp.gate_proj": (inter, hid), "mlp.up_proj": (inter, hid), "mlp.down_proj": (hid, inter)}
    w, k = {}, 64 * seed
    for i in range(case["layers"]):
        for name, shape in sizes.items():
            k += 1
            w[f"model.layers.{i}.{name}.weight"] = _fill(shape, k, dtype).mul_(0.02)
        for name in ("input_layernorm", "post_attention_layernorm"):
            w[f"model.layers.{i}.{name}.weight"] = torch.ones(hid, dtype=dtype, device=DEVICE)
    w["model.norm.weight"] = torch.ones(hid, dtype=dtype, device=DEVICE)
    w["model.embed_tokens.weight"] = _fill((case["vocab"], hid), 64 * seed, dtype)
    gen = torch.Generator().manual_seed(seed)
    follows = torch.randperm(case["vocab"], generator=gen).to(DEVICE)
    w["lm_head.weight"] = w["model.embed_tokens.weight"][follows] * 0.02
    gen = torch.Generator().manual_seed(seed + 1)
    lens = _sizes(case, seed)
    prompts = [torch.randint(0, case["vocab"], (n,), generator=gen).tolist() for n in lens]
    return w, prompts


def prepare(case, seed):
    from inferkernellab_amd import ops

    kind = case["kind"]
    if kind == "llama":
        from inferkernellab_amd.llama import LlamaConfig, LlamaForCausalLM, RotaryEmbedding

        w, prompts = _llama_weights(case, seed)
        cfg = LlamaConfig(vocab_size=case["vocab"], hidden_size=case["hidden"], intermediate_size=case["inter"],
                          num_hidden_layers=case["layers"], num_attention_heads=case["heads"],
                          num_key_value_heads=case["kv_heads"], head_dim=case["head_dim"])
        with torch.device("meta"):
            model = LlamaForCausalLM(cfg)
        model.load_state_dict(w, assign=True)
        model.model.rotary_emb = RotaryEmbedding(case["head_dim"], cfg.rope_theta).to(DEVICE)
        model.eval().requires_grad_(False)
        return {"case": case, "model": model, "prompts": prompts}
    if kind == "rope":
        raw = _rope_inputs(case, seed)
        from inferkernellab_amd import PagedKVCache

        dtype = DTYPES[case["dtype"]]
        fp8 = case["cache"] == "fp8"
        cache = PagedKVCache(raw["pool"], case["block"], case["kv_heads"], case["head_dim"],
                             dtype=torch.float8_e4m3fn if fp8 else dtype, act_dtype=dtype if fp8 else None,
                             device=DEVICE)
        for x in (cache.k, cache.v):
            x.view(torch.uint8).zero_()
        if fp8:
            cache.k_scale.fill_(1.0)
            cache.v_scale.fill_(1.0)
        return {"case": case, "cache": cache, "q_out": torch.empty_like(raw["q"]), **raw}
    raw = _inputs(case, seed)
    cache = _cache(case, raw)
    tables = raw["tables"]
    state = {"case": case, "cache": cache, "q": raw["q"], "tables": tables}
    if kind == "prefill":
        state["prefill"] = ops.PreparedPagedPrefill(cache, tables, raw["starts"], raw["ends"],
                                                    num_heads=case["heads"], query_width=raw["q"].shape[2])
        out = state["out"] = torch.empty_like(raw["q"])
        state["parts"] = _parts(out, raw)
        return state
    state["lens"], state["slots"] = raw["lens"], raw["slots"]
    state["new_k"], state["new_v"] = raw["new_k"].contiguous(), raw["new_v"].contiguous()
    if kind == "step":
        attention = ops.PreparedPagedAttention(raw["q"], cache, tables, raw["lens"], max_context_len=max(raw["ends"]))
        append = ops.PreparedAppend(state["new_k"], state["new_v"], cache, raw["slots"])
        state["step"] = ops.PreparedDecodeStep(attention, append)
    elif case["index"] == "i64":
        state["tables"], state["lens"] = tables.to(torch.int64), raw["lens"].to(torch.int64)
    return state


def run(state):
    from inferkernellab_amd import ops

    case = state["case"]
    kind = case["kind"]
    if kind == "step":
        return {"out": state["step"](), **_blocks(state["cache"], case["batch"])}
    if kind == "op":
        cache = state["cache"]
        ops.append_kv_hip(state["new_k"], state["new_v"], cache, state["slots"])
        out = ops.paged_decode_attention_hip_grouped(state["q"], cache, state["tables"], state["lens"])
        return {"out": out, **_blocks(cache, case["batch"])}
    if kind == "prefill":
        state["prefill"](state["q"], out=state["out"])
        return state["parts"]
    if kind == "rope":
        cache = state["cache"]
        q = ops.rope_append_kv_hip(state["q"], state["key"], state["value"], state["cos"], state["sin"], cache,
                                   state["slots"], query_out=state["q_out"])
        return {"q": q, **_blocks(cache, cache.layout.num_blocks)}
    from inferkernellab_amd.llama import LlamaPagedDecodeRunner

    dtype = torch.float8_e4m3fn if case["cache"] == "fp8" else None
    result = LlamaPagedDecodeRunner(state["model"], state["prompts"], max_new_tokens=case["new"],
                                    block_size=case["block"], max_num_batched_tokens=case["budget"],
                                    kv_cache_dtype=dtype).run()
    return {"prompt_logits": result.prompt_logits, "decode_logits": list(result.decode_logits),
            "tokens": torch.tensor(result.generated_tokens)}


# ------------------------------------------------------------ what is needed
def work(case):
    eb = 4 if case["dtype"] == "fp32" else 2
    h, hkv, d = case["heads"], case["kv_heads"], case["head_dim"]
    row = d + 4 if case["cache"] == "fp8" else d * eb  # one head's K or V row of a token in the cache
    if case["kind"] == "rope":
        t = case["tokens"]
        return {"bytes": t * (2 * h * d * eb + 2 * hkv * (d * eb + row) + 2 * d * eb + 4),
                "flops": t * (h + hkv) * d * 3}
    if case["kind"] == "llama":
        lens = _sizes(case, 0)
        hid = case["hidden"]
        layer = 2 * hid * h * d + 2 * hid * hkv * d + 3 * hid * case["inter"]
        weights = case["layers"] * layer + hid * case["vocab"]
        new, n = case["new"], len(lens)
        pairs = sum(x * (x + 1) // 2 + x * new + new * new // 2 for x in lens)
        prefill = sum(lens)
        batches = -(-prefill // case["budget"])
        kv = case["layers"] * hkv * row * 2
        return {"bytes": weights * eb * (new + batches) + kv * (prefill + sum(x * new for x in lens)),
                "flops": 2 * case["layers"] * layer * (prefill + n * new) + 2 * hid * case["vocab"] * n * (new + 1)
                + 4 * h * d * case["layers"] * pairs}
    sizes = _sizes(case, 0)
    if case["kind"] == "prefill":
        starts, spans = sizes
        pairs = sum(n * s + n * (n + 1) // 2 for s, n in zip(starts, spans))
        keys = sum(s + n for s, n in zip(starts, spans))
        return {"bytes": keys * hkv * row * 2 + sum(spans) * h * d * eb + case["batch"] * max(spans) * h * d * eb,
                "flops": pairs * h * 4 * d}
    b, idx = case["batch"], 8 if case["index"] == "i64" else 4
    table = sum(-(-n // case["block"]) for n in sizes) * idx
    append = 2 * b * hkv * (d * eb + row) + 4 * b
    return {"bytes": sum(sizes) * hkv * row * 2 + 2 * b * h * d * eb + table + b * idx + append,
            "flops": sum(sizes) * h * 4 * d}


def tolerance(case):
    # Attention outputs are rounded once to the query's type (half an ulp is
    # 2^-9 in bf16, 2^-12 in fp16) from fp32 accumulators, after
    # probabilities that may themselves be rounded to that type; FP8 codes
    # are given, not recomputed, except the new rows', where a value on a
    # rounding boundary may fall either way. A whole model passes such
    # differences through all its layers.
    if case["kind"] == "llama":
        return {"rel": 0.03, "max": 0.5, "differ": 0.01}
    rel = {"bf16": 1e-2, "fp16": 1.5e-3, "fp32": 5e-6}[case["dtype"]]
    return {"rel": rel, "max": 20 * rel, "differ": 1e-4}


# --------------------------------------------------------- results in 64 bits
def _wide(raw, case, name, blocks):
    """Rows of a request's blocks [tokens, kv heads, D] in 64 bits."""
    x = raw[name][blocks].double()
    if case["cache"] == "fp8":
        x = x * raw[name + "_scale"][blocks].double().unsqueeze(-1)
    return x.flatten(0, 1)


def _attend(q, k, v, start):
    """Causal attention in 64 bits: q [Hkv, G, T, D] at positions start..,
    k / v [Hkv, L, D]."""
    hkv, g, t, d = q.shape
    s = torch.bmm(q.reshape(hkv, g * t, d), k.transpose(1, 2).contiguous()).view(hkv, g, t, -1) * d**-0.5
    at = torch.arange(k.shape[1], device=q.device)
    seen = at.view(1, -1) <= start + torch.arange(t, device=q.device).view(-1, 1)
    p = torch.softmax(s.masked_fill(~seen, float("-inf")), dim=-1)
    return torch.bmm(p.view(hkv, g * t, -1), v).view(hkv, g, t, d)


def exact(case, seed):
    if case["kind"] == "rope":
        return _exact_rope(case, seed)
    if case["kind"] == "llama":
        return _exact_llama(case, seed)
    raw = _inputs(case, seed)
    h, hkv, d = case["heads"], case["kv_heads"], case["head_dim"]
    g = h // hkv
    out = torch.zeros(raw["q"].shape, dtype=torch.float64, device=DEVICE)
    for b, end in enumerate(raw["ends"]):
        blocks = raw["tables"][b, :raw["need"][b]].long()
        k = _wide(raw, case, "k", blocks)[:end].transpose(0, 1).contiguous()
        v = _wide(raw, case, "v", blocks)[:end].transpose(0, 1).contiguous()
        if case["kind"] != "prefill":
            q = raw["q"][b].double().view(hkv, g, 1, d)
            out[b] = _attend(q, k, v, end - 1).view(h, d)
            continue
        start, span = raw["starts"][b], end - raw["starts"][b]
        q = raw["q"][b, :, :span].double().view(hkv, g, span, d)
        for i in range(hkv):
            out[b, i * g:(i + 1) * g, :span] = _attend(q[i:i + 1], k[i:i + 1], v[i:i + 1], start)[0]
        out[b, :, span:] = v[:, 0].repeat_interleave(g, dim=0).unsqueeze(1)
    if case["kind"] == "prefill":
        return _parts(out, raw)
    # the appended rows
    res = {"out": out}
    slots, bs, n = raw["slots"].long(), case["block"], case["batch"]
    for name in ("k", "v"):
        new = raw["new_" + name]
        rows = raw[name][-n:].clone()
        at = slots // bs - (raw["pool"] - n)
        if case["cache"] == "fp8":
            codes, scale = _quantize(new)
            rows.view(torch.uint8)[at, slots % bs] = codes.view(torch.uint8)
            scales = raw[name + "_scale"][-n:].clone()
            scales[at, slots % bs] = scale
            res[name], res[name + "_scale"] = None, scales.transpose(1, 2).double()
        else:
            rows[at, slots % bs] = new
            res[name] = rows.double()
    return res


def _rotate(x, cos, sin):
    half = x.shape[-1] // 2
    return x * cos + torch.cat((-x[..., half:], x[..., :half]), dim=-1) * sin


def _exact_rope(case, seed):
    raw = _rope_inputs(case, seed)
    cos, sin = raw["cos"].double().unsqueeze(1), raw["sin"].double().unsqueeze(1)
    res = {"q": _rotate(raw["q"].double(), cos, sin)}
    if case["cache"] == "fp8":  # codes and their scales are whole values
        return {**res, "k": None, "k_scale": None, "v": None, "v_scale": None}
    for name, rows in (("k", _rotate(raw["key"].double(), cos, sin)), ("v", raw["value"].double())):
        full = torch.zeros((raw["pool"] * case["block"], *rows.shape[1:]), dtype=torch.float64, device=DEVICE)
        full[raw["slots"].long()] = rows
        res[name] = full.view(raw["pool"], case["block"], *rows.shape[1:])
    return res


def _exact_llama(case, seed):
    if case["cache"] == "fp8":
        return None  # the cache's rounding is part of the format
    w, prompts = _llama_weights(case, seed)
    h, hkv, d = case["heads"], case["kv_heads"], case["head_dim"]
    inv = 1.0 / (10000.0 ** (torch.arange(0, d, 2, dtype=torch.float64, device=DEVICE) / d))

    def norm(x, name):
        return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + 1e-6) * w[name].double()

    class Request:
        def __init__(self, prompt):
            self.ids, self.kv = prompt, [None] * case["layers"]

    def forward(requests, chunks):
        """Logits after each request's chunk of tokens; grows its K/V."""
        sizes = [len(c) for c in chunks]
        ids = torch.tensor([t for c in chunks for t in c], device=DEVICE)
        done = [0 if r.kv[0] is None else r.kv[0][0].shape[1] for r in requests]
        pos = torch.cat([torch.arange(s, s + n, device=DEVICE) for s, n in zip(done, sizes)]).double()
        angles = pos.view(-1, 1, 1) * inv
        cos, sin = torch.cat((angles, angles), -1).cos(), torch.cat((angles, angles), -1).sin()
        x = w["model.embed_tokens.weight"][ids].double()
        for i in range(case["layers"]):
            p = f"model.layers.{i}."
            y = norm(x, p + "input_layernorm.weight")
            q, k, v = (y @ w[p + f"self_attn.{n}_proj.weight"].double().t() for n in "qkv")
            q = _rotate(q.view(-1, h, d), cos, sin)
            k, v = _rotate(k.view(-1, hkv, d), cos, sin), v.view(-1, hkv, d)
            o, at = torch.empty_like(q), 0
            for r, n, s in zip(requests, sizes, done):
                kk, vv = (z[at:at + n].transpose(0, 1) for z in (k, v))
                if r.kv[i] is not None:
                    kk, vv = torch.cat((r.kv[i][0], kk), 1), torch.cat((r.kv[i][1], vv), 1)
                r.kv[i] = (kk, vv)
                qq = q[at:at + n].permute(1, 0, 2).reshape(hkv, h // hkv, n, d)
                o[at:at + n] = _attend(qq, kk, vv.contiguous(), s).reshape(h, n, d).transpose(0, 1)
                at += n
            x = x + o.reshape(-1, h * d) @ w[p + "self_attn.o_proj.weight"].double().t()
            y = norm(x, p + "post_attention_layernorm.weight")
            a, b = (y @ w[p + f"mlp.{n}_proj.weight"].double().t() for n in ("gate", "up"))
            x = x + (torch.nn.functional.silu(a) * b) @ w[p + "mlp.down_proj.weight"].double().t()
        last = torch.tensor(sizes, device=DEVICE).cumsum(0) - 1
        return norm(x[last], "model.norm.weight") @ w["lm_head.weight"].double().t()

    requests = [Request(p) for p in prompts]
    logits = torch.cat([forward([r], [r.ids]) for r in requests])
    prompt_logits, steps = logits, []
    for i in range(case["new"]):
        steps.append(logits)
        if i + 1 < case["new"]:
            logits = forward(requests, [[t] for t in logits.argmax(-1).tolist()])
    return {"prompt_logits": prompt_logits, "decode_logits": steps, "tokens": None}
