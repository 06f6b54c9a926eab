"""GPU: the pinned words of a context -- written by kernels, watched by the host -- when the context is dropped with a
step still queued, and when they are read under another stream than the step's."""
import weakref

import pytest
import torch

pytestmark = pytest.mark.gpu


def make_context(mi, dev):
    ctx = mi.DynamicInferenceContext(
        params_dtype=torch.bfloat16, num_layers=1, kv_channels=64, num_attention_heads=2, max_sequence_length=512,
        buffer_size_gb=0.01, buffer_guaranteed_fraction=0.0, max_requests_override=8, max_tokens_override=1024, device=dev)
    for i, n in enumerate((5, 300, 77)):
        ctx.add_request(i, torch.arange(n, device=dev), 20)
    return ctx


def keep_busy(dev, products=200):
    """Some 100 ms of work on the current stream (products of 1.1 TFLOP)."""
    a = torch.zeros(8192, 8192, dtype=torch.bfloat16, device=dev)
    for _ in range(products):
        torch.mm(a, a)


def test_words_of_a_dropped_context_are_not_handed_on(mi, dev):
    pinned = lambda: [torch.full((64,), 12345, dtype=torch.int32).pin_memory() for _ in range(4)]  # the words' block size
    ctx, other, spare = make_context(mi, dev), make_context(mi, dev), pinned()
    keep_busy(dev, 1)
    torch.cuda.synchronize()
    del other, spare                   # (what follows finds memory of every kind in the caches: an allocation may wait)
    keep_busy(dev)
    done = torch.cuda.Event()
    ctx.initialize_attention_state()   # its kernel waits behind the products
    done.record()
    words = ctx._counters.data_ptr()   # (the block's first; the maxima lie in it too)
    gone = weakref.ref(ctx)
    del ctx
    assert gone() is None
    rows = pinned()
    later = make_context(mi, dev)
    assert not done.query(), "the products ended too early to show anything"
    assert words not in [later._counters.data_ptr(), *(r.data_ptr() for r in rows)]
    later.initialize_attention_state()
    assert (later.max_seqlen_q, later.max_seqlen_k) == (300, 300)
    torch.cuda.synchronize()
    assert all((r == 12345).all() for r in rows)


def test_maxima_are_awaited_on_the_stream_that_makes_them(mi, dev):
    """Longer than the host watches a word without asking the stream (20 ms)."""
    ctx = make_context(mi, dev)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        keep_busy(dev)
        ctx.initialize_attention_state()
        done = torch.cuda.Event()
        done.record()
    assert not done.query(), "the products ended too early to show anything"
    assert (ctx.max_seqlen_q, ctx.max_seqlen_k) == (300, 300)
    torch.cuda.current_stream().wait_stream(side)
    ctx.update_requests(torch.ones(3, dtype=torch.uint8, device=dev), torch.zeros(3, dtype=torch.long, device=dev))
    ctx.initialize_attention_state()
    assert ctx.max_seqlen_q == 1 and ctx.active_token_count == 3


def test_a_word_that_never_comes_is_an_error(mi, dev):
    ctx = make_context(mi, dev)
    ctx._counters_host[5] = -1
    with pytest.raises(RuntimeError, match="without its results"):
        ctx._await(ctx._counters, 5, torch.cuda.current_stream())
