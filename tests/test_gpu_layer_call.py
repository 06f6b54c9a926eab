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


@pytest.mark.parametrize("lens,hidden,heads,cache,pad", [
    ([5], 6112, 8, None, 0),           # workgroups of 24 rows: the last workgroup's rows end beyond the matrix
    ([600], 4096, 32, None, 8),        # rows apart, the last one at the end of its storage
    ([3, 256], 5120, 64, None, 0),     # a matrix larger than what is read ahead
    ([3, 256], 5120, 64, "fp8_e4m3", 0),   # (nothing is read ahead)
    ([240] * 16, 2048, 16, None, 0),   # half of the workgroups have a span, or all
])
def test_reading_the_projection_ahead_changes_nothing(mi, dev, lens, hidden, heads, cache, pad):
    outs = []
    for by_module in (False, True):
        ctx = _context(mi, dev, lens, cache)
        ctx.update_requests(torch.ones(len(lens), dtype=torch.uint8, device=dev), torch.zeros(len(lens), dtype=torch.long, device=dev))
        ctx.initialize_attention_state()
        gen = torch.Generator(device=dev).manual_seed(2)
        layer = mi.PagedSelfAttentionLayer(2, hidden, heads, 2, 128, qk_norm="rms", device=dev).requires_grad_(False)
        for p in layer.parameters():
            p.normal_(0, 0.05, generator=gen)
        w = layer.linear_proj.weight
        room = torch.empty(w.numel() + (w.shape[0] - 1) * pad, dtype=w.dtype, device=dev)
        w.data = room.as_strided(w.shape, (w.shape[1] + pad, 1)).copy_(w.data)
        if by_module:
            layer.linear_qkv.register_forward_hook(lambda m, i, o: None)
        x = torch.empty(ctx.padded_active_token_count, 1, hidden, dtype=torch.bfloat16, device=dev).normal_(generator=gen)
        outs.append((layer(x, ctx)[0], ctx.memory_buffer))
    for a, b in zip(*outs):
        assert torch.equal(a, b)


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


@pytest.mark.parametrize("how", ["by the kernel", "large", "overridden"])
def test_update_leaves_the_mirrors_zero(mi, dev, how, monkeypatch):
    calls = []
    if how == "large":
        monkeypatch.setattr(mi.ops, "UPDATE_CLEARS_AT_MOST", 0)
    if how == "overridden":
        before = mi.DynamicInferenceContext.reset_attention_state
        monkeypatch.setattr(mi.DynamicInferenceContext, "reset_attention_state", lambda c: (calls.append(1), before(c))[1])
        class Other(mi.DynamicInferenceContext):
            def reset_attention_state(self):
                calls.append(2)
                super().reset_attention_state()
        monkeypatch.setattr(mi, "DynamicInferenceContext", Other)
    ctx = _context(mi, dev, [5, 256, 17, 300], None)
    finished = []
    for mask in ([1, 0, 1, 1], [1, 0, 1], [0, 0]):      # (the last empties the context)
        ctx._mirrors.fill_(7)
        calls.clear()
        ctx.update_requests(torch.tensor(mask, dtype=torch.uint8, device=dev), torch.arange(len(mask), device=dev))
        assert not ctx._mirrors.any() and ctx.block_table is None and (calls == [2, 1] or how != "overridden")
        finished.append(ctx.last_finished_request_ids)
        if ctx.total_request_count:
            ctx.initialize_attention_state()
    assert [f.numel() for f in finished] == [1, 1, 2] and sorted(torch.cat(finished).tolist()) == [0, 1, 2, 3]


@pytest.mark.parametrize("where", ["class", "object", "subclass"])
def test_a_replaced_reset_is_called(mi, dev, where, monkeypatch):
    """A reset put on the class itself, on one context or in a subclass runs after every update, as the class's own does."""
    calls = []
    own = mi.DynamicInferenceContext.reset_attention_state
    reset = lambda c: (calls.append(1), own(c))[1]
    if where == "class":
        monkeypatch.setattr(mi.DynamicInferenceContext, "reset_attention_state", reset)
    elif where == "subclass":
        monkeypatch.setattr(mi, "DynamicInferenceContext",
                            type("Other", (mi.DynamicInferenceContext,), {"reset_attention_state": reset}))
    ctx = _context(mi, dev, [5, 256, 17], None)
    if where == "object":
        ctx.reset_attention_state = lambda: reset(ctx)
    for mask in ([1, 0, 1], [0, 0]):      # (the last empties the context)
        ctx._mirrors.fill_(7)
        calls.clear()
        ctx.update_requests(torch.tensor(mask, dtype=torch.uint8, device=dev), torch.arange(len(mask), device=dev))
        assert calls == [1] and not ctx._mirrors.any() and ctx.block_table is None


@pytest.mark.parametrize("dtype", [torch.int32, torch.uint8])
@pytest.mark.parametrize("words", [0, 4, 4096 + 12])
def test_update_clears_the_rows_it_is_given_and_no_other(mi, dev, dtype, words):
    ctx = _context(mi, dev, [5, 256, 17], None)
    rows = torch.full((words + 8,), 7, dtype=torch.int32, device=dev)
    mirrors = ctx._mirrors.fill_(3).clone()
    mi.ops.update_requests(ctx, torch.tensor([1, 0, 1], dtype=dtype, device=dev), torch.arange(3, device=dev), rows[4:4 + words])
    torch.cuda.synchronize()
    assert ctx._counters_host.tolist()[:2] == [2, 0] and torch.equal(ctx._mirrors, mirrors)
    assert (rows[:4] == 7).all() and (rows[4 + words:] == 7).all() and not rows[4:4 + words].any()


DECODE_PARTS = ["core.forward_mixed_qkv", "class core.forward_mixed_qkv", "linear_qkv.forward", "linear_proj.forward",
                "ctx.fused_decode_step_attention", "class ctx.fused_decode_step_attention", "ctx.key_value_cache"]
PROMPT_PARTS = ["core._attend", "class core._attend", "ctx.fused_qkv_norm_rope_append",
                "class ctx.fused_qkv_norm_rope_append", "ctx.key_value_cache"]


@pytest.mark.parametrize("step,part", [("decode", p) for p in DECODE_PARTS] + [("prompts", p) for p in PROMPT_PARTS])
def test_replaced_parts_are_called(mi, dev, step, part, monkeypatch):
    """A part replaced on the object, on its class or in a subclass runs in a step that is otherwise folded into fewer
    calls, and the step's result is what it was."""
    lens = [3, 256, 40]
    owner, name = part.split()[-1].split(".")
    outs, calls = [], []
    for replaced in (False, True):
        ctx = _context(mi, dev, lens, None)
        if step == "decode":
            ctx.update_requests(torch.ones(3, dtype=torch.uint8, device=dev), torch.zeros(3, dtype=torch.long, device=dev))
            ctx.initialize_attention_state()
        gen = torch.Generator(device=dev).manual_seed(2)
        layer = mi.PagedSelfAttentionLayer(2, 512, 8, 2, 128, qk_norm="rms", device=dev).requires_grad_(False)
        for p in layer.parameters():
            p.normal_(0, 0.05, generator=gen)
        if replaced:
            target = ctx if owner == "ctx" else getattr(layer, owner)
            if part.startswith("class"):
                target = type(target)
            before = getattr(target, name)
            monkeypatch.setattr(target, name, lambda *a, **k: (calls.append(1), before(*a, **k))[1])
        table = mi.synthetic.rotary_angle_table(1024, 128, base=10000.0).to(dev)
        x = torch.empty(ctx.padded_active_token_count, 1, 512, dtype=torch.bfloat16, device=dev).normal_(generator=gen)
        outs.append(layer(x, ctx, (table, table))[0][:ctx.active_token_count].float())
    assert calls, "the replaced part was skipped"
    # (another kernel may do the step then: a rounding of the 16-bit result apart, a few of them after the projection)
    torch.testing.assert_close(outs[0], outs[1], rtol=2e-2, atol=2e-2)


def test_a_subclass_of_the_context_keeps_its_overrides(mi, dev):
    class Counting(mi.DynamicInferenceContext):
        steps = appends = 0

        def fused_decode_step_attention(self, *a, **k):
            self.steps += 1
            return super().fused_decode_step_attention(*a, **k)

        def fused_qkv_norm_rope_append(self, *a, **k):
            self.appends += 1
            return super().fused_qkv_norm_rope_append(*a, **k)

    ctx = Counting(params_dtype=torch.bfloat16, num_layers=1, kv_channels=128, num_attention_heads=2, max_sequence_length=1024,
                   buffer_size_gb=0.02, buffer_guaranteed_fraction=0.0, max_requests_override=4, max_tokens_override=1024, device=dev)
    layer = mi.PagedSelfAttentionLayer(1, 512, 8, 2, 128, device=dev).requires_grad_(False)
    for p in layer.parameters():
        p.zero_()
    ctx.add_request(0, torch.arange(70, device=dev), 20)
    for _ in range(2):
        ctx.initialize_attention_state()
        layer(torch.zeros(ctx.padded_active_token_count, 1, 512, dtype=torch.bfloat16, device=dev), ctx)
        ctx.update_requests(torch.ones(1, dtype=torch.uint8, device=dev), torch.zeros(1, dtype=torch.long, device=dev))
    assert (ctx.appends, ctx.steps) == (1, 1)


@pytest.mark.parametrize("cache", [None, "fp8_e4m3"], ids=["16bit", "fp8"])
def test_steps_do_not_see_what_callers_do_to_their_views(mi, dev, cache):
    ctx = _context(mi, dev, [5, 300], cache)
    for step in range(2):
        k, v, _ = ctx.key_value_cache(1)
        assert k.shape == v.shape == ctx.memory_buffer.shape[2:] and k.data_ptr() == ctx.memory_buffer.data_ptr()
        row = torch.full((ctx.padded_active_token_count, 1, 2, 128), 1.0 + step, dtype=torch.bfloat16, device=dev)
        ctx.append_key_value_cache(1, row, row)
        chunk, at = int(ctx.token_to_chunk_idx[0]), int(ctx.token_to_local_position_within_kv_chunk[0])
        scale = ctx.kv_scales[0, 0, chunk, 0] if cache else 1.0
        stored = k[chunk, at, 0, 0].view(torch.float8_e4m3fn) if cache else k[chunk, at, 0, 0]
        assert abs(float(stored) * float(scale) - (1.0 + step)) < 0.1
        k.unsqueeze_(0)
        v.transpose_(0, 1)
        for s in ctx.key_value_scales(1):
            if s is not None:
                s.unsqueeze_(0)
    with pytest.raises(IndexError):
        ctx.key_value_cache(3)
