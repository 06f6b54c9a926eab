"""Prompts from the QKV projection's output: keys and values appended by one call, queries normed and rotated by the tile
kernel -- against the separate calls (norm + rotary + append, then attention), whose own tests compare them with the oracle."""
import pytest
import torch

from oracle import paged_attention as oa
from oracle import rope_norm as orn

pytestmark = pytest.mark.gpu

CHUNK = 64


def _batch(mi, dev, lens, hq, hkv, d, dtype, pad, seed):
    gen = torch.Generator().manual_seed(seed)
    lens = torch.tensor(lens, dtype=torch.int32)
    T = int(lens.sum()) + pad
    table, n_chunks = mi.synthetic.build_block_table(lens, CHUNK, gen)
    cu = torch.zeros(len(lens) + 1, dtype=torch.int32)
    cu[1:] = torch.cumsum(lens, 0)
    pos, chunk, local = (x.to(torch.int64) for x in mi.synthetic.prefill_token_rows(cu, lens, table, CHUNK))
    tail = torch.zeros(pad, dtype=torch.int64)
    pos, local = torch.cat([pos, tail]), torch.cat([local, torch.arange(pad)])
    chunk = torch.cat([chunk, tail + n_chunks])           # padded rows: a chunk of their own
    mixed = torch.randn(T, 1, (hq + 2 * hkv) * d, generator=gen).to(dtype)
    weights = [(1 + 0.1 * torch.randn(d, generator=gen)).to(dtype).to(dev) for _ in range(2)]
    caches = [torch.zeros(n_chunks + 1, CHUNK, hkv, d, dtype=dtype, device=dev) for _ in range(2)]
    return [x.to(dev) for x in (mixed, pos, chunk, local, cu, lens, table)], weights, caches, int(lens.max())


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("hq,hkv,norm,interleaved,rope,lens,pad", [
    (8, 2, "rms", False, True, (2, 31, 33, 257, 300), 7),
    (6, 2, "l2", True, True, (65, 3, 129), 0),
    (32, 1, "none", False, True, (2,), 1),
    (20, 1, "rms", True, True, (515, 64), 0),
    (8, 8, "rms", False, False, (40, 700), 3),
    (4, 4, None, False, False, (5, 6, 7), 0),
])
def test_equals_the_separate_calls(mi, dev, dtype, d, hq, hkv, norm, interleaved, rope, lens, pad):
    (mixed, pos, chunk, local, cu, kv, table), (qw, kw), caches, longest = _batch(mi, dev, lens, hq, hkv, d, dtype, pad, d + hq)
    emb = mi.synthetic.rotary_angle_table(longest, d, base=10000.0).to(dev) if rope else None
    ref = [c.clone() for c in caches]
    T = mixed.size(0)
    query = torch.empty(T, 1, hq, d, dtype=dtype, device=dev)
    common = dict(num_query_heads=hq, num_kv_heads=hkv, norm=norm, rotary_emb=emb, q_positions=pos, k_positions=pos,
                  rotary_interleaved=interleaved, k_weight=kw if norm == "rms" else None, token_to_chunk_idx=chunk,
                  token_to_local_pos=local)
    qw = qw if norm == "rms" else None
    with mi.ops.tuning(norm_rope_vectorised=1):
        mi.ops.qkv_norm_rope_append(mixed, query_out=query, q_weight=qw, k_cache=ref[0], v_cache=ref[1], **common)
    want = mi.ops.paged_prefill_attention(query.squeeze(1), *ref, cu, kv, table, one_row_requests=False)

    assert mi.ops.qkv_prefill_supported(d, CHUNK, emb)
    cos_sin = mi.ops.qkv_key_append(mixed, k_cache=caches[0], v_cache=caches[1], **common)
    got = mi.ops.qkv_prefill_attention(mixed, *caches, cu, kv, table, num_query_heads=hq, num_kv_heads=hkv,
                                       max_kv_len=longest, cos_sin=cos_sin, q_weight=qw, norm=norm,
                                       rotary_interleaved=interleaved).squeeze(1)
    assert torch.equal(caches[1], ref[1])
    rel = lambda a, b: ((a.float() - b.float()).norm() / b.float().norm()).item()
    assert rel(caches[0], ref[0]) < 1e-3          # the norm's sum in another order: a rounding here and there
    assert rel(got, want) < (2e-3 if dtype == torch.bfloat16 else 5e-4)
    assert (got[int(kv.sum()):] == 0).all()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("hq,hkv,norm,interleaved,rope,lens,pad", [
    (8, 2, "rms", False, True, (2, 31, 33, 257, 300), 7),
    (6, 2, "l2", True, True, (65, 3, 129), 0),
    (20, 1, "rms", True, True, (515, 64), 0),
    (8, 8, None, False, False, (40, 200), 3),
])
def test_equals_the_oracle(mi, dev, dtype, d, hq, hkv, norm, interleaved, rope, lens, pad):
    """Values bit for bit; keys as the op-by-op chain (under 1 % differ at all, by at most two units in the last place of
    the head's largest: see the norm / rotary tests); attention within 2e-2 of fp32 attention over the oracle's cache."""
    (mixed, pos, chunk, local, cu, kv, table), (qw, kw), caches, longest = _batch(mi, dev, lens, hq, hkv, d, dtype, pad, d + hq)
    emb = orn.rotary_table(longest, d, interleaved=interleaved) if rope else None
    qw, kw = (qw, kw) if norm == "rms" else (None, None)
    eps = 1e-5 if norm == "rms" else 1e-6
    common = dict(num_query_heads=hq, num_kv_heads=hkv, norm=norm, eps=eps, rotary_interleaved=interleaved)
    cos_sin = mi.ops.qkv_key_append(mixed, k_cache=caches[0], v_cache=caches[1], k_weight=kw, q_positions=pos, k_positions=pos,
                                    rotary_emb=emb if emb is None else emb.to(dev), token_to_chunk_idx=chunk,
                                    token_to_local_pos=local, **common)
    got = mi.ops.qkv_prefill_attention(mixed, *caches, cu, kv, table, max_kv_len=longest, cos_sin=cos_sin, q_weight=qw,
                                       **common).squeeze(1).float().cpu()
    real = int(kv.sum())
    q, k, v = orn.split_mixed_qkv(mixed[:real].cpu(), hq, hkv)
    chain = dict(norm=norm, eps=eps, interleaved=interleaved)
    q = orn.norm_rope(q.reshape(real, hq, d), pos[:real].cpu(), emb, weight=qw if qw is None else qw.cpu(), **chain)
    k = orn.norm_rope(k.reshape(real, hkv, d), pos[:real].cpu(), emb, weight=kw if kw is None else kw.cpu(), **chain)
    v = v.reshape(real, hkv, d)
    at = (chunk[:real].cpu(), local[:real].cpu())
    assert torch.equal(caches[1].cpu()[at], v)
    keys = caches[0].cpu()[at]
    ulp = 2.0 ** (-7 if dtype == torch.bfloat16 else -10)
    err = (keys.float() - k.float()).abs()
    assert (keys != k).float().mean().item() < 0.01
    assert (err <= 2 * ulp * k.float().abs().amax(-1, keepdim=True)).all()
    kc, vc = (torch.zeros(c.shape, dtype=dtype) for c in caches)
    oa.kv_append(kc, vc, k, v, *at)
    ref = oa.paged_varlen_attention(q, kc, vc, cu.cpu(), kv.cpu(), table.cpu())
    assert (got[:real] - ref).abs().max().item() < 2e-2
    assert not got[real:].any()


@pytest.mark.parametrize("fp8", [False, True])
def test_core_takes_it_for_prompts_only(mi, dev, fp8, monkeypatch):
    """A step of fresh prompts goes through the two calls, one with a one-token prompt through the separate ones, with
    the same result."""
    calls = []
    real = mi.ops.qkv_prefill_attention
    monkeypatch.setattr(mi.ops, "qkv_prefill_attention", lambda *a, **k: calls.append(1) or real(*a, **k))
    hq, hkv, d = 8, 2, 128
    gen = torch.Generator(device=dev).manual_seed(3)
    emb = mi.synthetic.rotary_angle_table(400, d, base=10000.0).to(dev)
    core = mi.PagedSelfAttentionCore(1, d, qk_norm="rms", device=dev).requires_grad_(False)
    outs = {}
    for name, lens in (("fused", (70, 333)), ("separate", (70, 333)), ("one row", (70, 1))):
        ctx = mi.DynamicInferenceContext(
            params_dtype=torch.bfloat16, num_layers=1, kv_channels=d, num_attention_heads=hkv, max_sequence_length=400,
            buffer_size_gb=0.01, buffer_guaranteed_fraction=0.0, chunk_size_tokens=CHUNK, max_requests_override=4,
            kv_cache_dtype="fp8_e4m3" if fp8 else None)
        for i, n in enumerate(lens):
            ctx.add_request(i, torch.arange(n, device=dev))
        ctx.initialize_attention_state()
        gen.manual_seed(3)
        mixed = torch.randn(ctx.padded_active_token_count, 1, (hq + 2 * hkv) * d, generator=gen, device=dev).bfloat16()
        before = len(calls)
        if name == "separate":
            monkeypatch.setattr(ctx, "prefill_fusable", lambda *a: False)
        outs[name] = core.forward_mixed_qkv(mixed, hq, ctx, (emb, emb))
        assert (len(calls) > before) == (name == "fused")
        assert outs[name].isfinite().all()
    a, b = outs["fused"].float(), outs["separate"].float()
    assert ((a - b).norm() / b.norm()).item() < (1e-2 if fp8 else 3e-3)


def test_norm_weights_off_16_bytes_take_the_separate_calls(mi, dev):
    """A weight in the middle of one flat parameter buffer: taken anywhere by the separate calls, so taken here."""
    d, hq, hkv = 128, 8, 2
    outs = []
    for shift in (0, 1):
        core = mi.PagedSelfAttentionCore(1, d, qk_norm="rms", device=dev).requires_grad_(False)
        weights = torch.linspace(0.5, 1.5, 2 * d, device=dev).bfloat16()
        flat = torch.cat([weights[:shift], weights])
        core.q_layernorm_weight.data, core.k_layernorm_weight.data = flat[shift:shift + d], flat[shift + d:]
        assert (core.q_layernorm_weight.data_ptr() % 16 == 0) == (shift == 0)
        ctx = mi.DynamicInferenceContext(
            params_dtype=torch.bfloat16, num_layers=1, kv_channels=d, num_attention_heads=hkv, max_sequence_length=400,
            buffer_size_gb=0.01, buffer_guaranteed_fraction=0.0, chunk_size_tokens=CHUNK, max_requests_override=4)
        ctx.add_request(0, torch.arange(70, device=dev))
        ctx.initialize_attention_state()
        mixed = torch.randn(ctx.padded_active_token_count, 1, (hq + 2 * hkv) * d,
                            generator=torch.Generator(device=dev).manual_seed(3), device=dev).bfloat16()
        outs.append(core.forward_mixed_qkv(mixed, hq, ctx)[:70].float())
    assert ((outs[0] - outs[1]).norm() / outs[0].norm()).item() < 3e-3


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("d,hkv", [(128, 7), (128, 8), (128, 17), (64, 15), (64, 16), (128, 32)])
@pytest.mark.parametrize("T", [1, 2, 3, 4, 5, 9, 3072, 3073])
def test_keys_do_not_depend_on_the_tokens_beside_them(mi, dev, dtype, d, hkv, T):
    """A workgroup takes two tokens or four, by the heads and the call's length: either side of those lines, whole and partial
    workgroups give the bits of each token appended by itself."""
    (mixed, pos, chunk, local, *_), (_, kw), caches, longest = _batch(mi, dev, (T,), hkv, hkv, d, dtype, 0, d + T)
    emb = mi.synthetic.rotary_angle_table(longest, d, base=10000.0).to(dev)
    common = dict(num_query_heads=hkv, num_kv_heads=hkv, norm="rms", k_weight=kw, rotary_emb=emb)
    one, key = [c.clone() for c in caches], torch.empty(T, 1, hkv, d, dtype=dtype, device=dev)
    slots = lambda a, b: dict(token_to_chunk_idx=chunk[a:b], token_to_local_pos=local[a:b], q_positions=pos[a:b], k_positions=pos[a:b])
    cos_sin = mi.ops.qkv_key_append(mixed, k_cache=caches[0], v_cache=caches[1], **common, **slots(0, T))
    alone = [mi.ops.qkv_key_append(mixed[i:i + 1], k_cache=one[0], v_cache=one[1], **common, **slots(i, i + 1)) for i in range(T)]
    mi.ops.qkv_key_append(mixed, key_out=key, q_positions=pos, k_positions=pos, **common)
    assert torch.equal(caches[0], one[0]) and torch.equal(caches[1], one[1])
    assert torch.equal(cos_sin, torch.cat(alone))
    assert torch.equal(key.squeeze(1), caches[0][chunk, local])
