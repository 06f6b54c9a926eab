"""GPU: the attention layer's decode step as one native call against the same step module by module, and the
bookkeeping kernel with a mask of bytes against one of int32 -- bit for bit."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _context(mi, dev, lens, cache, dtype=torch.bfloat16):
    ctx = mi.DynamicInferenceContext(
        params_dtype=dtype, num_layers=2, kv_channels=128, num_attention_heads=2, max_sequence_length=1024,
        buffer_size_gb=0.02, buffer_guaranteed_fraction=0.0, max_requests_override=len(lens), max_tokens_override=4096,
        kv_cache_dtype=cache, device=dev)
    if cache is None:
        ctx.memory_buffer.normal_(generator=torch.Generator(device=dev).manual_seed(1))
    for i, n in enumerate(lens):
        ctx.add_request(i, torch.arange(n, device=dev), 400)
    ctx.initialize_attention_state()
    return ctx


@pytest.mark.parametrize("cache", [None, "fp8_e4m3"], ids=["16bit", "fp8"])
@pytest.mark.parametrize("lens", [[1], [3, 256, 40, 511, 512]])
def test_one_call_equals_the_modules(mi, dev, lens, cache):
    outs = []
    for by_module in (False, True):
        ctx = _context(mi, dev, lens, cache)
        ctx.update_requests(torch.ones(len(lens), dtype=torch.uint8, device=dev), torch.zeros(len(lens), dtype=torch.long, device=dev))
        ctx.initialize_attention_state()
        gen = torch.Generator(device=dev).manual_seed(2)
        layer = mi.PagedSelfAttentionLayer(2, 512, 8, 2, 128, qk_norm="rms", add_qkv_bias=True, device=dev).requires_grad_(False)
        for p in layer.parameters():
            p.normal_(0, 0.05, generator=gen)
        calls = []
        if by_module:  # a hook on a part makes the layer call it as a module
            layer.linear_qkv.register_forward_hook(lambda m, i, o: calls.append(1))
        table = mi.synthetic.rotary_angle_table(1024, 128, base=10000.0).to(dev)
        x = torch.empty(ctx.padded_active_token_count, 1, 512, dtype=torch.bfloat16, device=dev).normal_(generator=gen)
        out, bias = layer(x, ctx, (table, table))
        assert bias is None and out.shape == x.shape and len(calls) == by_module
        outs.append((out, ctx.memory_buffer, ctx.kv_scales))
    for a, b in zip(*outs):
        assert (a is None and b is None) or torch.equal(a, b)


def test_mask_of_bytes(mi, dev):
    lens = [5, 256, 17, 300, 1, 90]
    state = []
    for dtype in (torch.int32, torch.uint8):
        ctx = _context(mi, dev, lens, None)
        for mask in ([1, 1, 0, 1, 1, 1], [1, 0, 1, 1, 0], [1, 1, 1]):
            ctx.update_requests(torch.tensor(mask, dtype=dtype, device=dev),
                                torch.arange(len(mask), device=dev) + 7)
        state.append([ctx.total_request_count, ctx.chunk_allocator.chunk_count_avail, ctx.last_finished_request_ids.tolist(),
                      ctx.request_ids.tolist(), ctx.request_to_kv_chunk_ids.tolist(), ctx.token_to_input_ids[:4].tolist()])
    assert state[0] == state[1] and state[0][0] == 3
