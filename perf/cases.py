"""The work that users have this package do, as measurable cases.

Seven kinds, each called the way a program calls it:

* ``layer``   -- a decode step of one attention layer from hidden states to hidden states
                 (``PagedSelfAttentionLayer`` over a ``DynamicInferenceContext``): both projections, head norm, rotary
                 embedding, append and attention over the paged cache, 16-bit or fp8.
* ``attend``  -- a decode step by the calls of an unchanged ``Attention.forward``: ``append_key_value_cache``, then
                 ``flash_attn_with_kvcache``.
* ``prompts`` -- the first step of freshly admitted prompts of ragged lengths: ``PagedSelfAttentionCore`` on the QKV
                 projection's output.
* ``mixed``   -- chunks of prompts over an existing context together with one-token requests: norm, rotary embedding
                 and append in one call, then ``flash_attn_varlen_func``.
* ``mla``     -- a decode step over the latent cache of multi-latent attention.
* ``sample``  -- the tail of a step: one token drawn per row of logits and, on request, its log-probability.
* ``serve``   -- a serving loop on the host: prompts admitted, engine steps until every request has finished.

Lengths are drawn from the case itself, so that ``work`` knows them; values, block tables and prompts from the seed.
"""
import importlib
import math
import random
from types import SimpleNamespace

import torch

mi = importlib.import_module("megatron-mixtera_amd")

CHUNK = 256      # tokens of a KV chunk (latent caches: 64)
LATENT, LATENT_V = 576, 512


# ------------------------------------------------------------------------------------------------ the cases
def _layer(name, batch, max_requests, heads, kv_heads, d, hidden, lo, hi, cache="16bit", dtype="bf16", norm="rms"):
    return dict(name=name, kind="layer", batch=batch, max_requests=max_requests, heads=heads, kv_heads=kv_heads, d=d,
                hidden=hidden, lo=lo, hi=hi, cache=cache, dtype=dtype, norm=norm)


def _attend(name, batch, heads, kv_heads, d, lo, hi, dtype="bf16"):
    return dict(name=name, kind="attend", batch=batch, heads=heads, kv_heads=kv_heads, d=d, lo=lo, hi=hi, dtype=dtype)


def _prompts(name, batch, heads, kv_heads, d, lo, hi, cache="16bit", dtype="bf16", norm="rms"):
    return dict(name=name, kind="prompts", batch=batch, heads=heads, kv_heads=kv_heads, d=d, lo=lo, hi=hi, cache=cache,
                dtype=dtype, norm=norm)


def _mixed(name, prefill, new, ctx_lo, ctx_hi, decode, dec_lo, dec_hi, heads, kv_heads, d, dtype="bf16"):
    return dict(name=name, kind="mixed", prefill=prefill, new=new, ctx_lo=ctx_lo, ctx_hi=ctx_hi, decode=decode,
                dec_lo=dec_lo, dec_hi=dec_hi, heads=heads, kv_heads=kv_heads, d=d, dtype=dtype)


def _mla(name, batch, heads, lo, hi, dtype="bf16"):
    return dict(name=name, kind="mla", batch=batch, heads=heads, lo=lo, hi=hi, dtype=dtype)


def _sample(name, rows, vocab, top_k, top_p, peaked, log_probs, dtype="fp32"):
    return dict(name=name, kind="sample", rows=rows, vocab=vocab, top_k=top_k, top_p=top_p, peaked=peaked,
                log_probs=log_probs, dtype=dtype)


def _serve(name, requests, concurrent, prompt_lo, prompt_hi, gen_lo, gen_hi, layers, heads, kv_heads, d, hidden, vocab,
           top_k, top_p):
    return dict(name=name, kind="serve", requests=requests, concurrent=concurrent, prompt_lo=prompt_lo,
                prompt_hi=prompt_hi, gen_lo=gen_lo, gen_hi=gen_hi, layers=layers, heads=heads, kv_heads=kv_heads, d=d,
                hidden=hidden, vocab=vocab, top_k=top_k, top_p=top_p)


def listed():
    return [
        # one user in front of a chat: a single request, a few hundred tokens into the conversation
        _layer("layer_single_stream", 1, 4, 32, 8, 128, 4096, 777, 777),
        # the ordinary serving batch (benchmark configuration 2): 64 requests, contexts U[512, 8192]
        _layer("layer_batch64", 64, 64, 32, 8, 128, 4096, 512, 8192),
        # throughput serving over an fp8 cache (configuration 5): 256 requests, contexts U[1024, 32768]
        _layer("layer_batch256_fp8", 256, 256, 32, 8, 128, 4096, 1024, 32768, cache="fp8"),
        # a small model, few requests (configuration 1): 4 requests, 8/8 heads of 64, contexts U[64, 1024]
        _attend("attend_small_d64", 4, 8, 8, 64, 64, 1024),
        # long documents, a 70B-shaped layer (configuration 4): 16 requests of 131 072 tokens
        _attend("attend_long_context", 16, 64, 8, 128, 131072, 131072),
        # prompts of a small fp16 model with heads of 64 values, ragged lengths
        _prompts("prompts_ragged_d64_fp16", 11, 32, 8, 64, 33, 3001, dtype="fp16", norm="none"),
        # prompts into an fp8 cache, from a line to a long page
        _prompts("prompts_fp8_cache", 6, 32, 8, 128, 129, 4097, cache="fp8"),
        # continuous batching (configuration 3): 8 x 2048 new tokens over U[0, 4096] beside 120 decoding requests
        _mixed("mixed_prefill_decode", 8, 2048, 0, 4096, 120, 512, 8192, 32, 8, 128),
        # a chunk of a long document's prompt, 70B-shaped heads: 509 new tokens over some 60 000 cached ones
        _mixed("chunk_over_long_context", 1, 509, 61234, 61234, 0, 1, 1, 64, 8, 128),
        # multi-latent attention with 16 heads per rank, 64 requests
        _mla("mla_decode_16_heads", 64, 16, 512, 8192),
        # the draw at the end of a step: 64 rows of a 128k vocabulary, nucleus sampling
        _sample("sample_top_p", 64, 128256, 0, 0.9, False, False),
        # a small serving loop: 24 requests through 16 slots, prompts of a few dozen to a few hundred tokens
        _serve("serve_loop", 24, 16, 17, 301, 3, 16, 2, 32, 8, 128, 4096, 32000, 0, 0.9),
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


_MOST_BYTES, _MOST_FLOPS = 7.5e9, 0.7e12     # a drawn case costs no more than the largest listed ones


def draw(rng):
    while True:
        c = _draw_one(rng)
        w = work(c)
        if w["bytes"] <= _MOST_BYTES and w["flops"] <= (_MOST_FLOPS if c["kind"] != "mla" else 2 * _MOST_FLOPS):
            c.pop("name", None)
            return c


def _draw_one(rng):
    kind = rng.choice(("layer", "attend", "prompts", "mixed", "mla", "sample", "serve"))
    dtype = rng.choice(("bf16", "bf16", "fp16"))
    heads, kv_heads = rng.choice(((32, 8), (32, 8), (64, 8), (32, 4), (16, 2), (8, 8), (24, 8)))
    if kind == "layer":
        batch = _log_int(rng, 1, 256)
        hi = _log_int(rng, 64, 32768)
        cache = rng.choice(("16bit", "16bit", "fp8"))
        d = 128 if cache == "fp8" else rng.choice((64, 128, 128))
        return _layer("", batch, 4 * math.ceil(batch / 4), heads, kv_heads, d, rng.choice((2048, 4096, 5120)),
                      max(2, hi // rng.choice((1, 4, 16))), hi, cache, dtype, rng.choice(("rms", "none")))
    if kind == "attend":
        hi = _log_int(rng, 64, 131072)
        return _attend("", _log_int(rng, 1, 256), heads, kv_heads, rng.choice((64, 96, 128, 128, 256)),
                       max(2, hi // rng.choice((1, 4, 16))), hi, dtype)
    if kind == "prompts":
        hi = _log_int(rng, 33, 6000)
        cache = rng.choice(("16bit", "16bit", "fp8"))
        return _prompts("", _log_int(rng, 1, 16), heads, kv_heads, rng.choice((64, 128)), max(2, hi // rng.choice((1, 4, 16))),
                        hi, cache, dtype, rng.choice(("rms", "none")))
    if kind == "mixed":
        ctx = _log_int(rng, 64, 65536)
        dec = _log_int(rng, 64, 8192)
        return _mixed("", _log_int(rng, 1, 8), _log_int(rng, 17, 2048), ctx // rng.choice((1, 4)), ctx,
                      rng.choice((0, _log_int(rng, 1, 128))), max(2, dec // 4), dec, heads, kv_heads,
                      rng.choice((64, 128, 128, 256)), dtype)
    if kind == "mla":
        hi = _log_int(rng, 128, 65536)
        return _mla("", _log_int(rng, 1, 128), rng.choice((16, 32, 64, 128)), max(2, hi // rng.choice((1, 4, 16))), hi, dtype)
    if kind == "sample":
        top_k, top_p = rng.choice(((1, 0.0), (rng.randint(2, 200), 0.0), (0, round(rng.uniform(0.3, 0.98), 3)), (0, 0.0)))
        return _sample("", _log_int(rng, 1, 512), _log_int(rng, 32000, 152064), top_k, top_p, rng.random() < 0.5,
                       rng.random() < 0.3, rng.choice(("fp32", "bf16")))
    n = _log_int(rng, 2, 24)
    hi = _log_int(rng, 33, 400)
    top_k, top_p = rng.choice(((1, 0.0), (50, 0.0), (0, 0.9)))
    return _serve("", n, min(n, _log_int(rng, 2, 16)), max(2, hi // 8), hi, 2, rng.randint(4, 16), rng.choice((1, 2)), 32, 8,
                  rng.choice((64, 128)), 2048, 32000, top_k, top_p)


# ------------------------------------------------------------------------------------------------ sizes of a case
_DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}


def _lengths(n, lo, hi, salt):
    r = random.Random(n * 1_000_003 + lo * 1009 + hi * 31 + salt)
    return [r.randint(lo, hi) for _ in range(n)]


def _case_lengths(c):
    return _lengths(c["batch"], c["lo"], c["hi"], 1)


def _mixed_lengths(c):
    """(query lengths, kv lengths) of a mixed batch: the prompts' chunks first, then the one-token requests."""
    ctx = _lengths(c["prefill"], c["ctx_lo"], c["ctx_hi"], 2)
    dec = _lengths(c["decode"], c["dec_lo"], c["dec_hi"], 3)
    return [c["new"]] * c["prefill"] + [1] * c["decode"], [x + c["new"] for x in ctx] + dec


def _serve_plan(c):
    """(prompt length, tokens to generate) of every request."""
    return list(zip(_lengths(c["requests"], c["prompt_lo"], c["prompt_hi"], 4),
                    _lengths(c["requests"], c["gen_lo"], c["gen_hi"], 5)))


def _attention_work(q_lens, kv_lens, heads, kv_heads, dk, dv, kv_item, chunk=CHUNK, scales=False):
    """Bytes and operations of causal attention: keys and values in use once, queries in, results out, the table."""
    pairs = sum(q * (k - q) + q * (q + 1) // 2 for q, k in zip(q_lens, kv_lens))
    chunks = sum(-(-k // chunk) for k in kv_lens)
    nbytes = sum(kv_lens) * kv_heads * (dk + dv) * kv_item + sum(q_lens) * heads * (dk + dv) * 2 + chunks * 4 + len(kv_lens) * 4
    return nbytes + (chunks * kv_heads * 8 if scales else 0), 2 * heads * (dk + dv) * pairs


def work(case):
    c, kind = case, case["kind"]
    if kind == "layer":
        lens = _case_lengths(c)
        fp8 = c["cache"] == "fp8"
        b, f = _attention_work([1] * len(lens), lens, c["heads"], c["kv_heads"], c["d"], c["d"], 1 if fp8 else 2, scales=fp8)
        qkv, proj = (c["heads"] + 2 * c["kv_heads"]) * c["d"], c["heads"] * c["d"]
        return {"bytes": b - len(lens) * 4 * proj + c["hidden"] * (qkv + proj) * 2 + len(lens) * c["hidden"] * 4,
                "flops": f + 2 * len(lens) * c["hidden"] * (qkv + proj)}
    if kind == "attend":
        lens = _case_lengths(c)
        b, f = _attention_work([1] * len(lens), lens, c["heads"], c["kv_heads"], c["d"], c["d"], 2)
        return {"bytes": b + 4 * len(lens) * c["kv_heads"] * c["d"] * 2, "flops": f}
    if kind == "prompts":
        lens = _case_lengths(c)
        item = 1 if c["cache"] == "fp8" else 2
        # read the projection's output, write the cache and the result
        return {"bytes": sum(lens) * c["d"] * ((2 * c["heads"] + 2 * c["kv_heads"]) * 2 + 2 * c["kv_heads"] * item),
                "flops": _attention_work(lens, lens, c["heads"], c["kv_heads"], c["d"], c["d"], item)[1]}
    if kind == "mixed":
        q_lens, kv_lens = _mixed_lengths(c)
        b, f = _attention_work(q_lens, kv_lens, c["heads"], c["kv_heads"], c["d"], c["d"], 2)
        return {"bytes": b + sum(q_lens) * c["kv_heads"] * c["d"] * 4, "flops": f}
    if kind == "mla":
        lens = _case_lengths(c)
        b, f = _attention_work([1] * len(lens), lens, c["heads"], 0, LATENT, LATENT_V, 2, chunk=64)
        return {"bytes": b + sum(lens) * LATENT * 2 + len(lens) * LATENT * 2, "flops": f}
    if kind == "sample":
        n = c["rows"] * c["vocab"]
        return {"bytes": n * _DTYPES[c["dtype"]].itemsize + c["rows"] * 16, "flops": 4 * n}
    b = f = 0
    qkv, proj = (c["heads"] + 2 * c["kv_heads"]) * c["d"], c["heads"] * c["d"]
    plan = _serve_plan(c)
    steps = -(-sum(g for _, g in plan) // c["concurrent"])
    for p, g in plan:
        pb, pf = _attention_work([p] + [1] * (g - 1), [p] + [p + i for i in range(1, g)], c["heads"], c["kv_heads"], c["d"], c["d"], 2)
        b += c["layers"] * pb + g * c["vocab"] * 4
        f += c["layers"] * (pf + 2 * (p + g - 1) * c["hidden"] * (qkv + proj))
    return {"bytes": b + steps * c["layers"] * c["hidden"] * (qkv + proj) * 2, "flops": f}


def tolerance(case):
    """16-bit results carry a rounding or two of their own and one of the probabilities (2^-9 in bf16, 2^-12 in fp16);
    log-probabilities are 32-bit sums; tokens and bookkeeping are whole numbers."""
    if case["kind"] == "sample":
        return {"rel": 1e-5} if case["log_probs"] else "exact"
    return {"rel": 4e-3 if case.get("dtype") == "fp16" else 1e-2}


# ------------------------------------------------------------------------------------------------ inputs
def _device():
    return torch.device("cuda", torch.cuda.current_device())


def _generators(seed):
    """One generator on the host (tables, prompts) and one on the device (values)."""
    return torch.Generator().manual_seed(seed), torch.Generator(device=_device()).manual_seed(seed + 1)


def _randn(shape, dtype, gen, scale=1.0):
    return torch.empty(shape, dtype=dtype, device=_device()).normal_(0, scale, generator=gen)


def _angles(max_len, d):
    return mi.synthetic.rotary_angle_table(max_len, d, base=500000.0).to(_device())


def _context(c, lens, layers, max_len, *, max_requests, host, gen, dtype, fp8=False, latent=False):
    """A context whose pool holds these requests (and the reserve it keeps back), its free chunks in the shuffled order
    that a server reaches after a while, its cache filled with values ~ N(0, 1)."""
    chunk = 64 if latent else CHUNK
    need = sum(-(-n // chunk) for n in lens) + 2 * len(lens) + -(-max_len // chunk) + 4
    if latent:
        chunk_bytes = 2 * layers * chunk * LATENT
    else:
        chunk_bytes = (1 if fp8 else 2) * 2 * layers * chunk * c["kv_heads"] * c["d"] + (8 * layers * c["kv_heads"] if fp8 else 0)
    more = dict(cache_mla_latent=True, kv_lora_rank=LATENT_V, qk_pos_emb_head_dim=LATENT - LATENT_V) if latent else {}
    ctx = mi.DynamicInferenceContext(
        params_dtype=dtype, num_layers=layers, kv_channels=c.get("d", 128), num_attention_heads=c.get("kv_heads", 1),
        max_sequence_length=max_len, buffer_size_gb=(need + 0.5) * chunk_bytes / 1024**3, buffer_guaranteed_fraction=0.0,
        chunk_size_tokens=chunk, max_requests_override=max_requests, kv_cache_dtype="fp8_e4m3" if fp8 else None, **more)
    free = ctx.chunk_allocator.chunk_bag[:-1]
    free.copy_(free[torch.randperm(free.numel(), generator=host).to(free.device)])
    if not fp8:
        ctx.memory_buffer.normal_(0, 0.5 if latent else 1.0, generator=gen)
        return ctx
    for which in range(2):
        for layer in range(layers):
            pool, scales = ctx.memory_buffer[which, layer], ctx.kv_scales[which, layer]
            for a in range(0, pool.size(0), 2048):
                part = pool[a:a + 2048]
                mi.ops.quantize_chunks_fp8(_randn(part.shape, dtype, gen), part, scales[a:a + 2048])
    return ctx


def _decoding(ctx, lens, host):
    """Admit a prompt of ``len - 1`` tokens for every request and take one step: each request then decodes a token at
    position ``len - 1``."""
    dev = _device()
    tokens = torch.randint(0, 32000, (max(lens),), generator=host).to(dev)
    for i, n in enumerate(lens):
        ctx.add_request(i, tokens[:n - 1])
    ctx.initialize_attention_state()
    ctx.update_requests(torch.ones(len(lens), dtype=torch.int32, device=dev), tokens[:1].expand(len(lens)).contiguous())
    ctx.initialize_attention_state()
    return ctx


def _attention_layer(number, c, dtype, norm, gen):
    layer = mi.PagedSelfAttentionLayer(number, c["hidden"], c["heads"], c["kv_heads"], c["d"],
                                       qk_norm=None if norm == "none" else norm, dtype=dtype, device=_device())
    layer.requires_grad_(False)
    for linear in (layer.linear_qkv, layer.linear_proj):
        linear.weight.normal_(0, linear.input_size ** -0.5, generator=gen)
    _norm_weights(layer.core, gen)
    return layer


def _norm_weights(core, gen):
    core.requires_grad_(False)
    for w in (core.q_layernorm_weight, core.k_layernorm_weight):
        if w is not None:
            w.normal_(1.0, 0.02, generator=gen)


def prepare(case, seed):
    return _PREPARE[case["kind"]](case, seed)


def _prepare_layer(c, seed):
    host, gen = _generators(seed)
    dtype, lens = _DTYPES[c["dtype"]], _case_lengths(c)
    max_len = c["hi"] + 64
    ctx = _decoding(_context(c, lens, 1, max_len, max_requests=c["max_requests"], host=host, gen=gen, dtype=dtype,
                             fp8=c["cache"] == "fp8"), lens, host)
    hidden = torch.zeros(ctx.padded_active_token_count, 1, c["hidden"], dtype=dtype, device=_device())
    hidden[:len(lens)].normal_(0, 1, generator=gen)
    rope = _angles(max_len, c["d"])
    return dict(kind="layer", ctx=ctx, layer=_attention_layer(1, c, dtype, c["norm"], gen), hidden=hidden, rope=(rope, rope))


def _prepare_attend(c, seed):
    host, gen = _generators(seed)
    dtype, lens = _DTYPES[c["dtype"]], _case_lengths(c)
    ctx = _decoding(_context(c, lens, 1, c["hi"] + 64, max_requests=4 * math.ceil(len(lens) / 4), host=host, gen=gen,
                             dtype=dtype), lens, host)
    n = ctx.padded_active_token_count
    q, k, v = (torch.zeros(n, 1, h, c["d"], dtype=dtype, device=_device()) for h in (c["heads"], c["kv_heads"], c["kv_heads"]))
    for t in (q, k, v):
        t[:len(lens)].normal_(0, 1, generator=gen)
    return dict(kind="attend", ctx=ctx, q=q, k=k, v=v, scale=c["d"] ** -0.5)


def _prepare_prompts(c, seed):
    host, gen = _generators(seed)
    dtype, lens = _DTYPES[c["dtype"]], _case_lengths(c)
    max_len = c["hi"] + 64
    ctx = _context(c, lens, 1, max_len, max_requests=4 * math.ceil(len(lens) / 4), host=host, gen=gen, dtype=dtype,
                   fp8=c["cache"] == "fp8")
    tokens = torch.randint(0, 32000, (max(lens),), generator=host).to(_device())
    for i, n in enumerate(lens):
        ctx.add_request(i, tokens[:n])
    ctx.initialize_attention_state()
    mixed = torch.zeros(ctx.padded_active_token_count, 1, (c["heads"] + 2 * c["kv_heads"]) * c["d"], dtype=dtype, device=_device())
    mixed[:sum(lens)].normal_(0, 1, generator=gen)
    core = mi.PagedSelfAttentionCore(1, c["d"], qk_norm=None if c["norm"] == "none" else c["norm"], dtype=dtype, device=_device())
    _norm_weights(core, gen)
    rope = _angles(max_len, c["d"])
    return dict(kind="prompts", ctx=ctx, core=core, mixed=mixed, heads=c["heads"], rope=(rope, rope))


def _prepare_mixed(c, seed):
    host, gen = _generators(seed)
    dev, dtype = _device(), _DTYPES[c["dtype"]]
    q_lens, kv_lens = _mixed_lengths(c)
    table, n_chunks = mi.synthetic.build_block_table(torch.tensor(kv_lens, dtype=torch.int32), CHUNK, host)
    cu_q = torch.tensor([0] + q_lens, dtype=torch.int32).cumsum(0).to(torch.int32).to(dev)
    cu_k = torch.tensor([0] + kv_lens, dtype=torch.int64).cumsum(0).to(torch.int32).to(dev)
    lens, table = torch.tensor(kv_lens, dtype=torch.int32).to(dev), table.to(dev)
    position, chunk_idx, local = mi.synthetic.prefill_token_rows(cu_q, lens, table, CHUNK)
    total, d = sum(q_lens), c["d"]
    q, k, v = (_randn((total, h, d), dtype, gen) for h in (c["heads"], c["kv_heads"], c["kv_heads"]))
    cache = _randn((2, n_chunks, CHUNK, c["kv_heads"], d), dtype, gen)
    return dict(kind="mixed", q=q, k=k, v=v, q_out=torch.empty_like(q), cache=cache, table=table, cu_q=cu_q, cu_k=cu_k,
                lens=lens, position=position, chunk_idx=chunk_idx, local=local, max_q=max(q_lens), max_k=max(kv_lens),
                q_weight=1 + _randn((d,), dtype, gen, 0.02), k_weight=1 + _randn((d,), dtype, gen, 0.02),
                rope=_angles(max(kv_lens), d), scale=d ** -0.5)


def _prepare_mla(c, seed):
    host, gen = _generators(seed)
    dtype, lens = _DTYPES[c["dtype"]], _case_lengths(c)
    ctx = _decoding(_context(c, lens, 1, c["hi"] + 64, max_requests=4 * math.ceil(len(lens) / 4), host=host, gen=gen,
                             dtype=dtype, latent=True), lens, host)
    n = ctx.padded_active_token_count
    q = torch.zeros(n, 1, c["heads"], LATENT, dtype=dtype, device=_device())
    latent = torch.zeros(n, 1, LATENT, dtype=dtype, device=_device())
    q[:len(lens)].normal_(0, 1, generator=gen)
    latent[:len(lens)].normal_(0, 0.5, generator=gen)
    return dict(kind="mla", ctx=ctx, q=q, latent=latent, scale=0.072)


def _params(c):
    return SimpleNamespace(top_k=c["top_k"], top_p=c["top_p"], temperature=0.8, return_log_probs=False)


def _prepare_sample(c, seed):
    host, gen = _generators(seed)
    rows, vocab = c["rows"], c["vocab"]
    logits = _randn((rows, vocab), torch.float32, gen, 2.0 if c["peaked"] else 3.0)
    if c["peaked"]:  # a confident model: a few dozen tokens far above the rest
        at = torch.randint(0, vocab, (rows, 32), generator=gen, device=_device())
        logits.scatter_add_(1, at, torch.rand(rows, 32, generator=gen, device=_device()) * 6 + 9)
    return dict(kind="sample", logits=logits.to(_DTYPES[c["dtype"]]), vocab=vocab, params=_params(c), log_probs=c["log_probs"],
                uniform=torch.rand(rows, generator=gen, device=_device()))


def _prepare_serve(c, seed):
    host, gen = _generators(seed)
    dev, dtype = _device(), torch.bfloat16
    plan = _serve_plan(c)
    max_len = c["prompt_hi"] + c["gen_hi"]
    ctx = _context(c, [p + g for p, g in plan], c["layers"], max_len, max_requests=4 * math.ceil(c["concurrent"] / 4),
                   host=host, gen=gen, dtype=dtype)
    rope = _angles(max_len, c["d"])
    return dict(kind="serve", ctx=ctx, concurrent=c["concurrent"], vocab=c["vocab"], params=_params(c), rope=(rope, rope),
                layers=[_attention_layer(i + 1, c, dtype, "rms", gen) for i in range(c["layers"])],
                embedding=_randn((1024, c["hidden"]), dtype, gen),
                # the head is a table of the previous token's logits: the tokens drawn do not depend on roundings
                bigram=_randn((1024, c["vocab"]), torch.float32, gen, 3.0),
                prompts=[(torch.randint(0, 1024, (p,), generator=host).to(dev), g) for p, g in plan],
                uniform=torch.rand(sum(g for _, g in plan) + 1, c["concurrent"], generator=gen, device=dev))


_PREPARE = {"layer": _prepare_layer, "attend": _prepare_attend, "prompts": _prepare_prompts, "mixed": _prepare_mixed,
            "mla": _prepare_mla, "sample": _prepare_sample, "serve": _prepare_serve}


# ------------------------------------------------------------------------------------------------ one pass
def run(state):
    return _RUN[state["kind"]](state)


def _run_layer(s):
    out, _ = s["layer"](s["hidden"], s["ctx"], s["rope"])
    return _with_cache({"out": out}, s["ctx"])


def _with_cache(outputs, ctx):
    outputs["cache"] = ctx.memory_buffer
    if ctx.kv_scales is not None:
        outputs["scales"] = ctx.kv_scales
    return outputs


def _run_attend(s):
    ctx = s["ctx"]
    ctx.append_key_value_cache(1, s["k"], s["v"])
    k_cache, v_cache, table = ctx.key_value_cache(1)
    out = mi.flash_attn_with_kvcache(q=s["q"], k_cache=k_cache, v_cache=v_cache, cache_seqlens=ctx.kv_seq_lengths,
                                     causal=True, block_table=table, softmax_scale=s["scale"])
    return {"out": out, "cache": ctx.memory_buffer}


def _run_prompts(s):
    return _with_cache({"out": s["core"].forward_mixed_qkv(s["mixed"], s["heads"], s["ctx"], s["rope"])}, s["ctx"])


def _run_mixed(s):
    k_cache, v_cache = s["cache"][0], s["cache"][1]
    mi.ops.norm_rope_append(s["q"], s["k"], value=s["v"], query_out=s["q_out"], norm="rms", q_weight=s["q_weight"],
                            k_weight=s["k_weight"], rotary_emb=s["rope"], q_positions=s["position"], k_positions=s["position"],
                            k_cache=k_cache, v_cache=v_cache, token_to_chunk_idx=s["chunk_idx"], token_to_local_pos=s["local"])
    out = mi.flash_attn_varlen_func(s["q_out"], k_cache, v_cache, s["cu_q"], s["cu_k"], s["max_q"], s["max_k"],
                                    softmax_scale=s["scale"], causal=True, block_table=s["table"], seqused_k=s["lens"])
    return {"out": out, "query": s["q_out"], "cache": s["cache"]}


def _run_mla(s):
    ctx = s["ctx"]
    ctx.append_key_value_cache(1, s["latent"], None)
    cache, _, table = ctx.key_value_cache(1)
    out = mi.flash_decode_and_prefill(s["q"], cache, None, ctx.max_seqlen_q, ctx.max_seqlen_k, None, None,
                                      ctx.kv_seq_lengths, table, softmax_scale=s["scale"], mla_head_dim_v=LATENT_V)
    return {"out": out, "cache": ctx.memory_buffer}


def _run_sample(s):
    tokens = mi.sampling.sample_from_logits(s["logits"], s["params"], s["vocab"], uniform=s["uniform"])
    if s["log_probs"]:
        return {"tokens": tokens, "log_probs": mi.ops.selected_log_probs(s["logits"], tokens)}
    return {"tokens": tokens}


def _run_serve(s):
    ctx, last = s["ctx"], []

    def forward_step(input_ids, position_ids):
        ids = input_ids[0] % 1024
        hidden = s["embedding"][ids].unsqueeze(1)
        for layer in s["layers"]:
            hidden = hidden + layer(hidden, ctx, s["rope"])[0]
        last.append(ctx.last_token_logits(hidden.transpose(0, 1)))     # the rows that a head takes
        return s["bigram"][ctx.last_token_logits(ids.to(torch.int32).view(1, -1, 1)).view(-1).long()].unsqueeze(0)

    tokens, finished, admitted, step = [], [], 0, 0
    ctx.reset()
    while admitted < len(s["prompts"]) or ctx.has_unfinished_requests():
        while admitted < len(s["prompts"]) and ctx.total_request_count < s["concurrent"]:
            prompt, budget = s["prompts"][admitted]
            ctx.add_request(admitted, prompt, budget)
            admitted += 1
        n = ctx.total_request_count - ctx.paused_request_count
        got = mi.step.generate_output_tokens_dynamic_batch(ctx, forward_step, s["params"], -1, vocab_size=s["vocab"],
                                                           uniform=s["uniform"][step, :n])
        tokens.append(got["sample"])
        finished.append(got["finished_request_ids"])
        step += 1
    return {"tokens": torch.cat(tokens), "finished": torch.cat(finished), "last_hidden": torch.cat(last),
            "cache": ctx.memory_buffer[:, :, :ctx.dummy_chunk_idx]}


_RUN = {"layer": _run_layer, "attend": _run_attend, "prompts": _run_prompts, "mixed": _run_mixed, "mla": _run_mla,
        "sample": _run_sample, "serve": _run_serve}
