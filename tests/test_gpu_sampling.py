"""GPU: last-token gather, sampling and the finished-request mask (through the C ABI).

Bars.  The gather, the argmax, the top-k cut and the mask are integer / selection work: equality
with the checker.  The top-p cut and the draw depend on sums of exponentials, which the kernel
carries as 2^-32 fixed point and the checker in fp64: a result must equal the checker's whenever
the checker's decision has a margin (2e-6 of the total mass: the
kernel's exponentials are fp32), and must in every case satisfy the definition within that margin
(mass strictly above the cut <= top_p < mass down to the cut; CDF bracket of the drawn index).
"""
import math
from types import SimpleNamespace

import pytest
import torch

from oracle import sampling as osm

pytestmark = pytest.mark.gpu

TOL = 2e-6        # top-p cut: distance of the kept mass from top_p
DRAW_TOL = 2e-6   # draw: distance of u from the CDF steps either side of the drawn index


def _logits(R, V, seed, dtype=torch.float32, spread=3.0):
    g = torch.Generator().manual_seed(seed)
    return (torch.randn(R, V, generator=g) * spread).to(dtype)


def _with_negative_nan(x, where):
    """A copy with NaNs whose sign is set (a conversion may drop a NaN's sign, so the bits are written in the type)."""
    bits = {torch.float32: -0x400000, torch.bfloat16: -0x40, torch.float16: -0x200}[x.dtype]   # 0xffc00000, 0xffc0, 0xfe00
    whole = torch.int32 if x.dtype == torch.float32 else torch.int16
    return x.contiguous().view(whole).masked_fill(where, bits).view(x.dtype)


def _by_one_workgroup(mi, y, u, top_k, top_p, temperature=0.7):
    """(tokens, cuts) of the form that walks a row with one workgroup: without a workspace, and for draws from rows that would fit
    the registers of a workgroup as the first part of a wider row, masked from there on."""
    lib, (R, V) = mi._lib.load(), y.shape
    if top_k != 1 and V <= 65536:
        wide = torch.full((R, 65544), float("-inf"), dtype=y.dtype, device=y.device)
        wide[:, :V] = y
        y = wide
    token = torch.empty(R, dtype=torch.int64, device=y.device)
    cut = torch.empty(R, dtype=torch.float32, device=y.device)
    code = {torch.float32: 0, torch.bfloat16: 1, torch.float16: 2}[y.dtype]
    rc = lib.mi_sample_from_logits(y.data_ptr(), y.stride(0), code, R, y.size(1), top_k, top_p, temperature, u.data_ptr(), 0,
                                   token.data_ptr(), cut.data_ptr(), None, None, None, -1, None,
                                   torch.cuda.current_stream().cuda_stream)
    assert rc == 0, lib.mi_last_error()
    return token, cut


# ----------------------------------------------------------------------------------------------
# last-token gather
# ----------------------------------------------------------------------------------------------
@pytest.mark.parametrize("dtype,E", [(torch.bfloat16, 4096), (torch.float32, 1000), (torch.bfloat16, 37),
                                     (torch.float32, 128256), (torch.bfloat16, 3)])
def test_last_token_gather_bit_exact(mi, dev, dtype, E):
    g = torch.Generator().manual_seed(E)
    q_lens = torch.randint(1, 40, (300,), generator=g, dtype=torch.int32)
    q_lens[5:150] = 1
    if E > 100000:
        q_lens = q_lens[:12]
    T = int(q_lens.sum()) + 7  # padding rows at the end
    rows = torch.randn(T, E, generator=g).to(dtype).to(dev)
    got = mi.ops.last_token_gather(rows, q_lens.to(dev))
    want = rows.cpu()[osm.last_token_indices(q_lens)]
    assert got.dtype == dtype and torch.equal(got.cpu(), want)


def test_last_token_gather_strided_source(mi, dev):
    g = torch.Generator().manual_seed(3)
    q_lens = torch.tensor([4, 1, 9, 2], dtype=torch.int32)
    big = torch.randn(16, 96, generator=g).bfloat16().to(dev)
    rows = big[:, 8:72]  # row stride 96, offset 16 bytes
    got = mi.ops.last_token_gather(rows, q_lens.to(dev))
    assert torch.equal(got.cpu(), rows.cpu()[osm.last_token_indices(q_lens)])
    assert mi.ops.last_token_gather(rows, q_lens[:0].to(dev)).shape == (0, 64)


# ----------------------------------------------------------------------------------------------
# greedy
# ----------------------------------------------------------------------------------------------
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("V", [1, 63, 1000, 32000, 128256])
def test_greedy_is_first_argmax(mi, dev, dtype, V):
    x = _logits(9, V, V, dtype)
    if V >= 63:
        x[1, :] = 0.5                      # all equal -> index 0
        x[2, 40] = x[2].max()              # two equal maxima -> the lower index
        x[2, 7] = x[2, 40]
        x[3, 10] = 0.0
        x[3, 20] = -0.0                    # signed zeros compare equal
        x[3] = torch.where(x[3] > 0, -x[3], x[3])
        x[3, 10], x[3, 20] = -0.0, 0.0
        x[4, V - 1] = 1e4                  # last element
        x[5, 5] = float("inf")
        x[6, :] = float("-inf")
    s, mask = mi.ops.sample_from_logits(x.to(dev), top_k=1)
    assert mask is None and s.dtype == torch.int64
    assert torch.equal(s.cpu(), osm.sample_from_logits(x, top_k=1))


# ----------------------------------------------------------------------------------------------
# filters
# ----------------------------------------------------------------------------------------------
def _check_draw(x_scaled, cut, u, s):
    """CDF bracket of every drawn index for the kept set {x >= cut}; returns the fp64 probabilities."""
    keep = x_scaled >= cut[:, None]
    pr = osm.kept_probabilities(x_scaled, keep)
    cdf = pr.cumsum(-1)
    R = x_scaled.size(0)
    idx = torch.arange(R)
    assert keep[idx, s].all(), "a filtered entry was drawn"
    assert (pr[idx, s] > 0).all()
    hi = cdf[idx, s]
    lo = hi - pr[idx, s]
    want = u.double()
    assert ((lo - DRAW_TOL <= want) & (want <= hi + DRAW_TOL)).all()
    exact = osm.draw_inverse_cdf(pr, u)
    clear = ((want - lo).abs() > DRAW_TOL) & ((hi - want).abs() > DRAW_TOL)
    assert clear.any() and torch.equal(s[clear], exact[clear])
    return pr


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("V,k", [(64, 2), (1000, 50), (32000, 40), (128256, 2), (128256, 50), (128256, 5000),
                                 (777, 777)])
@pytest.mark.parametrize("temperature", [1.0, 0.7])
def test_top_k_cut_is_exact_and_draw_brackets(mi, dev, dtype, V, k, temperature):
    R = 16
    x = _logits(R, V, 7 * V + k, dtype)
    if V > 100:
        x[3, 100:100 + min(60, V - 100)] = x[3].float().topk(k).values[-1]  # many ties at the k-th value
        x[4, V // 2:] = float("-inf")  # pre-masked entries
    if k > V // 2:
        x[4] = _logits(1, V, 5, dtype)[0]
    u = torch.rand(R, generator=torch.Generator().manual_seed(k))
    s, _, cut = mi.ops.sample_from_logits(x.to(dev), top_k=k, temperature=temperature, uniform=u.to(dev),
                                          return_cut=True)
    xs = osm.scaled_logits(x, temperature)
    kth = torch.topk(xs, k, dim=-1).values[:, -1]
    assert torch.equal(cut.cpu(), kth)
    _check_draw(xs, kth, u, s.cpu())
    # the same call again gives the same tokens (integer sums)
    s2, _ = mi.ops.sample_from_logits(x.to(dev), top_k=k, temperature=temperature, uniform=u.to(dev))
    assert torch.equal(s, s2)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("V", [50, 1000, 32000, 128256])
@pytest.mark.parametrize("top_p", [0.05, 0.5, 0.9, 0.999])
def test_top_p_cut_meets_the_definition(mi, dev, dtype, V, top_p):
    R = 16
    spread = 3.0 if V < 100000 else 4.0
    x = _logits(R, V, 11 * V + int(top_p * 1000), dtype, spread)
    x[2] *= 0.05           # nearly flat row: the prefix is long
    x[5, V // 3:] = float("-inf")
    u = torch.rand(R, generator=torch.Generator().manual_seed(V))
    _check_top_p(mi, dev, x, top_p, 0.9, u)


def _check_top_p(mi, dev, x, top_p, temperature, u):
    s, _, cut = mi.ops.sample_from_logits(x.to(dev), top_p=top_p, temperature=temperature, uniform=u.to(dev),
                                          return_cut=True)
    cut = cut.cpu()
    xs = osm.scaled_logits(x, temperature)
    pr = xs.double().softmax(-1)
    above = (pr * (xs > cut[:, None])).sum(-1)          # mass strictly above the cut value
    down_to = (pr * (xs >= cut[:, None])).sum(-1)       # ... including it
    assert (above <= top_p + TOL).all() and (down_to > top_p - TOL).all()
    # equality with the checker's kept set wherever its decision is not within the margin
    keep = osm.top_p_keep(xs, top_p)
    want_cut = xs.masked_fill(~keep, float("inf")).min(-1).values
    clear = ((above - top_p).abs() > TOL) & ((down_to - top_p).abs() > TOL)
    assert torch.equal(cut[clear], want_cut[clear])
    _check_draw(xs, cut, u, s.cpu())


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("top_p", [0.3, 0.9])
def test_top_p_one_pass_form_and_its_fallbacks(mi, dev, dtype, top_p):
    """Top-p on rows of 32 768: peaked rows find their cut among the listed candidates, the others (flat, nearly
    flat, a few finite values, half the row tied at the top) go through the general path; both must meet the
    definition."""
    V = 32768
    x = _logits(10, V, 1200 + int(10 * top_p), dtype, spread=5.0)   # rows 7-9: peaked random rows
    x[0, :] = -0.75
    x[1, :] = float("-inf"); x[1, [5, 17000, 32767]] = torch.tensor([0.5, 1.5, 1.0], dtype=dtype)
    x[2, :] = 0.25; x[2, 12345] = 9.0
    x[3, : V // 2] = 3.0
    x[4, ::2] = float("-inf")
    x[5] = (torch.arange(V).float() / V * 30).to(dtype)
    x[6] *= 0.02
    u = torch.rand(10, generator=torch.Generator().manual_seed(int(100 * top_p)))
    _check_top_p(mi, dev, x, top_p, 1.0, u)


def test_no_filter_draws_from_the_full_softmax(mi, dev):
    x = _logits(32, 5000, 21)
    u = torch.rand(32, generator=torch.Generator().manual_seed(22))
    s, _, cut = mi.ops.sample_from_logits(x.to(dev), temperature=1.3, uniform=u.to(dev), return_cut=True)
    assert torch.isinf(cut).all() and (cut < 0).all()
    _check_draw(osm.scaled_logits(x, 1.3), cut.cpu(), u, s.cpu())
    # top_p = 1 filters nothing either
    s1, _ = mi.ops.sample_from_logits(x.to(dev), top_p=1.0, temperature=1.3, uniform=u.to(dev))
    assert torch.equal(s1, s)


@pytest.mark.parametrize("mode", [dict(top_k=6), dict(top_p=0.8), dict()])
def test_draw_frequencies_follow_the_kept_probabilities(mi, dev, mode):
    V, n = 48, 1 << 16
    row = _logits(1, V, 31)[0]
    x = row.expand(n, V).contiguous()
    u = torch.rand(n, generator=torch.Generator().manual_seed(32))
    s, _ = mi.ops.sample_from_logits(x.to(dev), uniform=u.to(dev), **mode)
    if "top_k" in mode:
        keep = osm.top_k_keep(row[None], mode["top_k"])
    elif "top_p" in mode:
        keep = osm.top_p_keep(row[None], mode["top_p"])
    else:
        keep = torch.ones(1, V, dtype=torch.bool)
    pr = osm.kept_probabilities(row[None], keep)[0]
    freq = torch.bincount(s.cpu(), minlength=V).double() / n
    assert (freq[~keep[0]] == 0).all()
    sigma = (pr * (1 - pr) / n).sqrt()
    assert ((freq - pr).abs() <= 5 * sigma + 1e-6).all()


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("k", [2, 10, 200, 256, 257, 768, 769])
def test_top_k_one_pass_form_and_its_fallbacks(mi, dev, dtype, k):
    """Rows of 32 768 and a small k take the form that lists candidates above a sampled threshold in one pass; rows
    where the estimate cannot work -- flat (every value a candidate), a few finite values (fewer candidates than k),
    a spike in an otherwise flat row, half the row tied at the maximum -- must come out the same through the general
    path.  k = 769 never takes the one-pass form."""
    V = 32768
    x = _logits(10, V, 900 + k, dtype)
    x[0, :] = -0.75                                             # flat: every entry equals the cut
    x[1, :] = float("-inf"); x[1, [5, 17000, 32767]] = torch.tensor([0.5, 1.5, 1.0], dtype=dtype)  # three finite values
    x[2, :] = 0.25; x[2, 12345] = 9.0                           # one spike over a flat row
    x[3, : V // 2] = 3.0                                        # half the row tied at the top
    x[4, ::2] = float("-inf")                                   # every other entry pre-masked
    x[5] = (torch.arange(V).float() / V).to(dtype)              # sorted ascending: the sample sees every level
    x[6] = (torch.arange(V, 0, -1).float() / V).to(dtype)
    u = torch.rand(10, generator=torch.Generator().manual_seed(k))
    s, _, cut = mi.ops.sample_from_logits(x.to(dev), top_k=k, uniform=u.to(dev), return_cut=True)
    xs = osm.scaled_logits(x, 1.0)
    kth = torch.topk(xs, k, dim=-1).values[:, -1]
    assert torch.equal(cut.cpu(), kth)
    _check_draw(xs, kth, u, s.cpu())
    assert s[1].item() in (5, 17000, 32767) and (k > 1 and s[2].item() >= 0)
    s2, _ = mi.ops.sample_from_logits(x.to(dev), top_k=k, uniform=u.to(dev))
    assert torch.equal(s, s2)


def test_extreme_rows(mi, dev):
    V = 4096
    x = _logits(6, V, 41)
    x[0, :] = 1.25                       # flat row: every entry equals the cut, all are kept
    x[1, 9] = float("inf")               # no distribution: argmax
    x[2, 100] = 80.0                     # one entry holds all the mass
    x[3, :] = float("-inf"); x[3, 77] = 0.0
    x[4, 5] = float("nan")               # NaN counts as the maximum, as in torch.argmax
    u = torch.tensor([0.5, 0.3, 0.9999, 0.2, 0.1, 0.7])
    for mode in (dict(top_k=10), dict(top_p=0.9), dict()):
        s, _ = mi.ops.sample_from_logits(x.to(dev), uniform=u.to(dev), **mode)
        s = s.cpu()
        assert s[0].item() == int(0.5 * V) or abs(s[0].item() - 0.5 * V) <= 1
        assert s[1].item() == 9 and s[2].item() == 100 and s[3].item() == 77 and s[4].item() == 5
        assert 0 <= s[5].item() < V
    # clamp to the tokenizer's vocabulary (sampling path only)
    x = _logits(64, 300, 42)
    u = torch.rand(64, generator=torch.Generator().manual_seed(43))
    s, _ = mi.ops.sample_from_logits(x.to(dev), uniform=u.to(dev))
    sc, _ = mi.ops.sample_from_logits(x.to(dev), uniform=u.to(dev), vocab_size=100)
    assert torch.equal(sc, s.clamp(0, 99)) and (s > 99).any()


def test_argument_errors(mi, dev):
    x = _logits(4, 100, 51).to(dev)
    u = torch.rand(4).to(dev)
    with pytest.raises(mi._lib.KernelError, match="top-k is larger"):
        mi.ops.sample_from_logits(x, top_k=101, uniform=u)
    with pytest.raises(mi._lib.KernelError, match="both greater than zero"):
        mi.ops.sample_from_logits(x, top_k=5, top_p=0.5, uniform=u)
    with pytest.raises(mi._lib.KernelError, match="temperature"):
        mi.ops.sample_from_logits(x, temperature=0.0, uniform=u)
    with pytest.raises(ValueError, match="uniform"):
        mi.ops.sample_from_logits(x, top_k=5)
    with pytest.raises(ValueError):
        mi.ops.sample_from_logits(x.double(), top_k=1)
    with pytest.raises(RuntimeError, match="no CPU path"):
        mi.ops.sample_from_logits(x.cpu(), top_k=1)
    s, m = mi.ops.sample_from_logits(x[:0], top_k=1)
    assert s.numel() == 0


# ----------------------------------------------------------------------------------------------
# the reference's surface and the finished-request mask
# ----------------------------------------------------------------------------------------------
def test_sample_from_logits_surface(mi, dev):
    x = _logits(8, 2000, 61).to(dev)
    params = SimpleNamespace(top_k=1, top_p=0.0, temperature=1.0)
    assert torch.equal(mi.sampling.sample_from_logits(x, params).cpu(), x.cpu().argmax(-1))
    before = x.clone()
    params = SimpleNamespace(top_k=0, top_p=0.9, temperature=0.8)
    g = torch.Generator(device=dev).manual_seed(5)
    a = mi.sampling.sample_from_logits(x, params, vocab_size=2000, generator=g)
    g.manual_seed(5)
    b = mi.sampling.sample_from_logits(x, params, vocab_size=2000, generator=g)
    assert torch.equal(a, b) and torch.equal(x, before)
    with pytest.raises(AssertionError, match="both greater than zero"):
        mi.sampling.sample_from_logits(x, SimpleNamespace(top_k=2, top_p=0.5, temperature=1.0))
    with pytest.raises(AssertionError, match="larger than vocab size"):
        mi.sampling.sample_from_logits(x, SimpleNamespace(top_k=50, top_p=0.0, temperature=1.0), vocab_size=50)
    with pytest.raises(AssertionError):
        mi.sampling.sample_from_logits(x, SimpleNamespace(top_k=2.0, top_p=0.0, temperature=1.0))


def test_decode_step_tail_on_a_context(mi, dev):
    """logits -> last-token rows -> sample + mask -> update_requests, against the checker."""
    Ctx = mi.DynamicInferenceContext
    c = Ctx(params_dtype=torch.bfloat16, num_layers=1, kv_channels=16, num_attention_heads=2,
            max_sequence_length=128, buffer_size_gb=0.01, buffer_guaranteed_fraction=0.1, chunk_size_tokens=16,
            device=dev)
    g = torch.Generator().manual_seed(71)
    V, term = 500, 3
    prompts = [5, 17, 1, 30, 9, 2]
    budgets = [3, 50, 2, 40, 1, 60]   # requests 0, 2 and 4 run out of length soon
    for i, (n, b) in enumerate(zip(prompts, budgets)):
        c.add_request(i, torch.randint(10, V, (n,), generator=g).to(dev), num_tokens_to_generate=b)
    for step in range(3):
        c.initialize_attention_state()
        T = c.padded_active_token_count
        logits = (torch.randn(1, T, V, generator=g) * 3).bfloat16().to(dev)
        if step == 1:
            logits[0, :, term] = 50.0  # everyone draws the termination id
        n = c.total_request_count - c.paused_request_count
        act = slice(c.paused_request_count, c.total_request_count)
        q_lens = c.request_query_lengths[act].cpu()
        last = c.last_token_logits(logits)
        assert torch.equal(last.cpu(), logits[0].cpu()[osm.last_token_indices(q_lens)])
        u = torch.rand(n, generator=g)
        params = SimpleNamespace(top_k=4, top_p=0.0, temperature=1.0)
        sample, mask = mi.sampling.sample_and_finish_mask(c, last, params, term, vocab_size=V, uniform=u.to(dev))
        want = osm.sample_from_logits(last.cpu(), top_k=4, uniform=u, vocab_size=V)
        assert torch.equal(sample.cpu(), want)
        want_mask = osm.active_request_mask(want, term, c.request_kv_length_offsets[act].cpu(), q_lens,
                                            c.request_output_lengths[act].cpu())
        assert mask.dtype == torch.uint8 and torch.equal(mask.cpu(), want_mask)
        if step == 0:
            assert want_mask.tolist().count(0) >= 1  # the one-token budget ends here
        c.update_requests(mask, sample.clone())
        if step == 1:
            assert not c.has_unfinished_requests()
            break


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("V", [1, 7, 4096, 32003, 131072])
def test_selected_log_probs_match_fp64_checker(mi, dev, dtype, V):
    """log_softmax(row)[id] with one read of the row: 2e-5 absolute against fp64 (fp32 sums of up to
    131 072 terms, hardware exp2 / log)."""
    g = torch.Generator().manual_seed(V)
    T = 37
    x = (torch.randn(T, V, generator=g) * 5).to(dtype)
    if V > 64:
        x[1, 10:40] = float("-inf")
        x[2, :] = 3.0                         # uniform row: -log V
        x[3, V // 2] = 60.0                   # one dominant entry
    ids = torch.randint(0, V, (T,), generator=g)
    if V > 64:
        ids[3] = V // 2
    got = mi.ops.selected_log_probs(x.to(dev), ids.to(dev)).cpu()
    want = osm.selected_log_probs(x, ids)
    assert torch.isfinite(got).all()
    assert (got.double() - want).abs().max().item() <= 2e-5
    if V > 64:
        assert abs(got[2].item() + float(torch.tensor(float(V)).log())) <= 2e-5
        assert abs(got[3].item()) <= 2e-5


def test_selected_log_probs_unaligned_rows_and_bad_ids(mi, dev):
    g = torch.Generator().manual_seed(5)
    big = torch.randn(6, 1003, generator=g)
    x = big[:, 1:1002]                         # rows neither 16-byte aligned nor a multiple of 4 wide
    ids = torch.randint(0, 1001, (6,), generator=g)
    got = mi.ops.selected_log_probs(x.to(dev)[:, :], ids.to(dev)).cpu()
    xd = big.to(dev)[:, 1:1002]
    got2 = mi.ops.selected_log_probs(xd, ids.to(dev)).cpu()
    want = osm.selected_log_probs(x, ids)
    assert (got.double() - want).abs().max().item() <= 2e-5
    assert (got2.double() - want).abs().max().item() <= 2e-5
    ids[4] = 1001
    ids[5] = -1
    bad = mi.ops.selected_log_probs(xd, ids.to(dev)).cpu()
    assert torch.isnan(bad[4]) and torch.isnan(bad[5]) and torch.isfinite(bad[:4]).all()


def test_context_log_probs_through_the_kernel(mi, dev):
    """calculate_log_probs on a mixed step: ids from the shifted prompt, grouped per request."""
    Ctx = mi.DynamicInferenceContext
    saved = (Ctx.TOKEN_ROUNDER, Ctx.REQUEST_ROUNDER)
    try:
        Ctx.TOKEN_ROUNDER, Ctx.REQUEST_ROUNDER = 4, 4
        ctx = Ctx(params_dtype=torch.bfloat16, num_layers=1, kv_channels=64, num_attention_heads=2,
                  max_sequence_length=64, buffer_size_gb=0.01, buffer_guaranteed_fraction=0.1, chunk_size_tokens=16,
                  max_requests_override=16, max_tokens_override=256, device=dev)
        g = torch.Generator().manual_seed(8)
        V = 300
        prompts = [torch.randint(0, V, (n,), generator=g) for n in (5, 1, 9)]
        for rid, pr in enumerate(prompts):
            ctx.add_request(rid, pr.to(dev), num_tokens_to_generate=4)
        ctx.initialize_attention_state()
        T = ctx.padded_active_token_count        # 15 active rows padded to 16
        logits = torch.randn(1, T, V, generator=g)
        new = torch.randint(0, V, (3,), generator=g)
        got = ctx.calculate_log_probs(logits.to(dev), new.to(dev))
        ids = osm.scored_token_ids(torch.cat(prompts), torch.tensor([5, 1, 9]), new)
        want = osm.selected_log_probs(logits[0][: ctx.active_token_count], ids)
        assert [len(r) for r in got] == [5, 1, 9]
        flat = torch.tensor([v for r in got for v in r], dtype=torch.float64)
        assert (flat - want).abs().max().item() <= 2e-5
        # last-token rows only
        rows = ctx.last_token_logits(logits.to(dev))
        got_last = ctx.calculate_log_probs(rows.unsqueeze(0), new.to(dev), only_last_token_logits=True)
        want_last = osm.selected_log_probs(logits[0][osm.last_token_indices(torch.tensor([5, 1, 9]))], new)
        assert (torch.tensor(got_last, dtype=torch.float64).flatten() - want_last).abs().max().item() <= 2e-5
    finally:
        Ctx.TOKEN_ROUNDER, Ctx.REQUEST_ROUNDER = saved


@pytest.mark.parametrize("R,V", [(1, 16384), (2, 16389), (5, 50257), (64, 32000), (85, 49152), (128, 65536), (129, 65536), (1, 260000),
                                 (32, 24577), (3, 32768), (64, 32769), (16, 57345), (7, 65537), (86, 65539), (257, 57344)])
@pytest.mark.parametrize("kind", ["flat", "peaked", "equal", "few", "masked", "nan"])
def test_rows_in_parts_equal_rows_by_one_workgroup(mi, dev, R, V, kind):
    """Rows cut into parts, and rows in the registers of a workgroup, give the tokens and cut values of the workgroup that walks a
    row, bit for bit: where their estimates hold, and where they fail (equal values, a handful of values, most of the row
    masked).  Sizes either side of the lines between the forms."""
    g = torch.Generator().manual_seed(R + V)
    x = torch.randn(R, V, generator=g) * 3
    if kind == "peaked":
        x[:, torch.randint(0, V, (20,), generator=g)] += 15
    elif kind == "equal":
        x.fill_(-2.5)
    elif kind == "few":
        x = torch.randint(0, 4, (R, V), generator=g).float()
    elif kind == "masked":
        x[:, ::2], x[:, 1::3] = float("-inf"), -1e9
    elif kind == "nan":
        x[R // 2, V // 3] = float("nan")
    u = torch.rand(R, generator=g).to(dev)
    for dtype in (torch.float32, torch.bfloat16):
        y = x.to(dtype).to(dev)
        for top_k, top_p in ((1, 0.0), (0, 0.0), (0, 0.5), (0, 0.95), (0, 1.0), (2, 0.0), (50, 0.0), (768, 0.0), (769, 0.0)):
            got, _, cut = mi.ops.sample_from_logits(y, top_k=top_k, top_p=top_p, temperature=0.7, uniform=u, return_cut=True)
            want, want_cut = _by_one_workgroup(mi, y, u, top_k, top_p)
            assert torch.equal(got, want), (dtype, top_k, top_p)
            assert torch.equal(cut, want_cut), (dtype, top_k, top_p)


@pytest.mark.parametrize("V", [1000, 16387, 80001])
@pytest.mark.parametrize("mode", [dict(top_p=0.3), dict(top_p=0.9), dict(), dict(top_k=5)])
def test_logits_too_large_for_masses_take_the_argmax(mi, dev, V, mode):
    """From some 4e8 on, the product with log2(e) rounds by more than the exponent's range and the maximum's own mass may be
    zero: such rows have no distribution, and no element that a uniform number could fall on."""
    g = torch.Generator().manual_seed(V)
    x = (torch.randn(8, V, generator=g) * 1e30).to(dev)
    u = torch.rand(8, generator=g).to(dev)
    got, _ = mi.ops.sample_from_logits(x, uniform=u, temperature=0.7, **mode)
    kept = (x * (1 / 0.7)).amax(-1, keepdim=True) * (1 - 1e-6)   # (a maximum with a mass: itself and what rounds with it)
    assert (x.gather(1, got[:, None]) * (1 / 0.7) >= kept).all()


@pytest.mark.parametrize("R,V,pad", [(3, 16387, 0), (128, 80001, 1), (86, 140000, 4), (5, 30011, 2), (40, 1003, 3), (6, 50001, 1)])
@pytest.mark.parametrize("kind", ["rising", "negative", "zeros", "huge", "wide", "negative nan", "part masked", "all masked", "infinite"])
def test_parts_where_the_bins_are_at_their_edges(mi, dev, R, V, pad, kind):
    """Draws from rows in parts, and in the registers of a workgroup, against one workgroup that walks a row: a maximum that rises
    from batch to batch of a part (the bins move), values whose integer order is not theirs, values that leave the bins'
    range, parts of nothing but -inf or NaN, rows off 16 bytes."""
    g = torch.Generator().manual_seed(R + V)
    x = torch.randn(R, V, generator=g) * 3
    if kind == "rising":
        x += torch.arange(V) * 1e-3
    elif kind == "negative":
        x = -x.abs() - 1e-3
    elif kind == "zeros":
        x = torch.where(x > 4, -torch.zeros(1), torch.where(x > 2, torch.zeros(1), -x.abs()))
    elif kind == "huge":
        x *= 1e30
    elif kind == "wide":
        x *= 200
    negative_nan = torch.zeros(R, V, dtype=torch.bool)
    if kind == "negative nan":
        negative_nan[:, ::7] = True
        negative_nan[R // 2] = True
    elif kind == "part masked":
        x[:, : V // 2] = float("-inf")
        negative_nan[R // 2, : V // 2] = True
    elif kind == "all masked":
        x[::2] = float("-inf")
    elif kind == "infinite":
        x[R // 2, V // 3] = float("inf")
    u = torch.rand(R, generator=g).to(dev)
    for dtype in (torch.float32, torch.bfloat16):
        y = torch.zeros(R, V + pad, dtype=dtype, device=dev)[:, :V]
        y.copy_(_with_negative_nan(x.to(dtype), negative_nan))
        for top_k, top_p in ((0, 0.0), (0, 0.3), (0, 0.9), (0, 0.999), (2, 0.0), (300, 0.0)):
            got, _, cut = mi.ops.sample_from_logits(y, top_k=top_k, top_p=top_p, temperature=0.7, uniform=u, return_cut=True)
            want, want_cut = _by_one_workgroup(mi, y, u, top_k, top_p)
            rows = ((~negative_nan).sum(-1) >= max(top_k, 1)).to(dev)   # (below that, the masked end of the wider row is above the NaNs)
            assert torch.equal(got[rows], want[rows]), (dtype, top_k, top_p)
            assert torch.equal(cut[rows], want_cut[rows]), (dtype, top_k, top_p)


@pytest.mark.parametrize("V", [1 << 18, 1 << 20])
@pytest.mark.parametrize("first,last", [(0.5028, 5.9754), (0.5183, 5.9913)], ids=["truncated", "rounded"])
def test_the_window_holds_the_cut_of_a_wide_row(mi, dev, V, first, last):
    """The wider the row, the coarser the units in which a part's bins are summed (2^-11 of a value at 2^20): most of the mass
    here lies at two values whose weights would be furthest apart after truncating, or are after rounding, the cut within 1e-5
    of the edge between two bins that hold 1e-3 each.  Both have to be listed; otherwise one workgroup walks the row several
    times, for the same token."""
    lib = mi._lib.load()
    value = lambda bins: (1.0 - bins) / 64      # `bins` below the upper edge of the first bin, whose number is 0
    a, c1, c2, d = (value(f) for f in (first, 3.5, 4.5, last))
    few = V // 1000
    n_a = int((V - 2 * few) / (1 + math.exp(a - d)))    # as much mass in the first level as in the last
    x = torch.full((V,), d)
    x[:n_a], x[n_a:n_a + few], x[n_a + few:n_a + 2 * few] = a, c1, c2
    w = x.double().exp()
    top_p = float(w[:n_a + few].sum() / w.sum()) + 1e-5
    x = x[torch.randperm(V, generator=torch.Generator().manual_seed(V))].view(1, V).to(dev)
    u = torch.full((1,), 0.37, device=dev)
    room = torch.zeros(lib.mi_sample_workspace_bytes(1, V, 0, top_p), dtype=torch.uint8, device=dev)
    got = []
    for ws, size in ((room.data_ptr(), room.numel()), (None, 0)):
        token = torch.empty(1, dtype=torch.int64, device=dev)
        cut = torch.empty(1, dtype=torch.float32, device=dev)
        rc = lib.mi_sample_from_logits_ws(x.data_ptr(), V, 0, 1, V, 0, top_p, 1.0, u.data_ptr(), 0, token.data_ptr(), cut.data_ptr(),
                                          None, None, None, -1, None, ws, size, torch.cuda.current_stream().cuda_stream)
        assert rc == 0, lib.mi_last_error()
        got.append((token.item(), cut.item()))
    assert got[0] == got[1] and got[0][1] == torch.tensor(c2, dtype=torch.float32).item()
    # (the workspace: four rows of a word per part, each on a line of 256 bytes; the last counts what the parts listed)
    parts = min(V // 4096, 64)
    assert room[768:768 + 4 * parts].view(torch.int32).sum().item() == 2 * few


@pytest.mark.parametrize("buffer", ["whole", "off a line", "too small", "on the host", "empty"])
def test_sampling_inside_use_workspace(mi, dev, buffer):
    """A buffer for attention's scratch that does not serve the parts of the rows is passed over, not refused."""
    gen = torch.Generator().manual_seed(11)
    logits = torch.randn(8, 65536, generator=gen).to(dev)
    u = torch.rand(8, generator=gen).to(dev)
    want, _ = mi.ops.sample_from_logits(logits, top_p=0.9, uniform=u)
    big = torch.empty(64 << 20, dtype=torch.uint8, device=dev)
    given = {"whole": big, "off a line": big[16:], "too small": big[:4096], "empty": big[:0],
             "on the host": torch.empty(64 << 20, dtype=torch.uint8)}[buffer]
    with mi.ops.use_workspace(given):
        got, _ = mi.ops.sample_from_logits(logits, top_p=0.9, uniform=u)
    assert torch.equal(got, want)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("R,V", [(129, 65537), (257, 70001), (1024, 65540), (1025, 65540)])
def test_top_p_of_many_wide_rows(mi, dev, R, V, dtype):
    """More than 128 rows that do not fit the registers of a workgroup: one part each up to 1 024 rows, a walk from there on.  The
    same tokens and cuts as the walk's: flat, peaked and equal rows, half masked ones, rows with a NaN."""
    lib = mi._lib.load()
    gen = torch.Generator(device=dev).manual_seed(R)
    x = torch.empty(R, V, device=dev).normal_(0, 3, generator=gen)
    x[1::8, 7::997] += 14
    x[2::8] = -2.5
    x[3::8, ::2] = float("-inf")
    x[4::32, V // 3] = float("nan")
    x[5::8] = x[5::8].round()
    x[6::8, : V - 9] = float("-inf")
    y = x.to(dtype)
    del x
    u = torch.rand(R, device=dev, generator=gen)
    assert (lib.mi_sample_workspace_bytes(R, V, 0, 0.9) > 0) == (R <= 1024)
    for top_p in (0.3, 0.9, 0.999, 1.0):
        got, _, cut = mi.ops.sample_from_logits(y, top_p=top_p, temperature=0.7, uniform=u, return_cut=True)
        want, want_cut = _by_one_workgroup(mi, y, u, 0, top_p)
        assert torch.equal(got, want) and torch.equal(cut, want_cut), top_p


@pytest.mark.parametrize("short,off", [(1, 0), (0, 16)], ids=["too small", "off a line"])
def test_many_rows_pass_over_a_workspace_that_does_not_serve(mi, dev, short, off):
    """More than 128 rows did without scratch at every size before they had a use for it: a buffer that does not serve is not used
    and not written.  128 rows refuse it, as they did."""
    lib, V = mi._lib.load(), 65537
    gen = torch.Generator(device=dev).manual_seed(3)
    for R in (128, 129):
        y = torch.empty(R, V, device=dev).normal_(0, 3, generator=gen)
        u = torch.rand(R, device=dev, generator=gen)
        room = torch.full((lib.mi_sample_workspace_bytes(R, V, 0, 0.9) + 256,), 0x5a, dtype=torch.uint8, device=dev)
        token = torch.empty(R, dtype=torch.int64, device=dev)
        rc = lib.mi_sample_from_logits_ws(y.data_ptr(), V, 0, R, V, 0, 0.9, 0.7, u.data_ptr(), 0, token.data_ptr(), None, None, None, None,
                                          -1, None, room.data_ptr() + off, room.numel() - 256 - short,
                                          torch.cuda.current_stream().cuda_stream)
        assert (rc == 0) == (R > 128)
        if rc == 0:
            assert torch.equal(token, _by_one_workgroup(mi, y, u, 0, 0.9)[0])
        assert (room == 0x5a).all()


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("V", [4, 8, 9, 255, 4097, 16391, 32767, 32768, 32769, 65535, 65536])
def test_rows_in_the_registers_of_a_workgroup(mi, dev, V, dtype):
    """Rows that start on any element and end within a group of 16 bytes; wavefronts without elements (short rows), the widest
    rows of either number of groups; lists of a few members, of many, and none that holds the cut (equal values, a top-k that
    ends far below the bins)."""
    R = 129 if V > 32768 else 7     # (the rows of a wide filter that are not done in parts)
    x = _logits(R, V, V, torch.float32)
    x[6] *= 60 if V % 2 else 3000   # (the k-th value far below the bins, and below the wider ones)
    x[1, V // 2:] = -90.0
    x[2] = x[2, 0]
    if V > 200:
        x[3, 100:180] = x[3].topk(40).values[-1]
        x[4, ::3] = float("-inf")
        x[5, V - 1] = 30.0
    y = torch.zeros(R, V + 3, dtype=dtype, device=dev)[:, 1:V + 1]
    y.copy_(x)
    u = torch.rand(R, generator=torch.Generator().manual_seed(V))
    u[5] = 0.999
    ud = u.to(dev)
    xs = osm.scaled_logits(y.cpu(), 0.8)
    for mode in (dict(), dict(top_k=2), dict(top_k=min(50, V)), dict(top_k=V - 1), dict(top_p=0.5), dict(top_p=0.97)):
        s, _, cut = mi.ops.sample_from_logits(y, temperature=0.8, uniform=ud, return_cut=True, **mode)
        s, cut = s.cpu(), cut.cpu()
        if "top_k" in mode:
            assert torch.equal(cut, torch.topk(xs, mode["top_k"], dim=-1).values[:, -1]), mode
        elif "top_p" in mode:
            pr = osm.kept_probabilities(xs, torch.ones_like(xs, dtype=torch.bool))
            above = torch.where(xs > cut[:, None], pr, 0).sum(-1)
            upto = torch.where(xs >= cut[:, None], pr, 0).sum(-1)
            assert (above <= mode["top_p"] + TOL).all() and (upto > mode["top_p"] - TOL).all(), mode
        else:
            assert torch.isinf(cut).all()
        _check_draw(xs, cut, u, s)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("V", [17, 1000, 16389, 32768, 50000])
def test_a_top_k_above_the_count_of_numbers_keeps_them_all(mi, dev, V, dtype):
    """NaNs with their sign set lie below -inf.  Where the top k reach down to them every number is kept, and the token is that of
    the plain draw from the numbers, masked tokens (the first among them) never."""
    x = _logits(5, V, V, dtype)
    x[:, 0] = float("-inf")
    negative_nan = torch.zeros(5, V, dtype=torch.bool)
    negative_nan[0, V // 2] = True
    negative_nan[1, 1::3] = True
    negative_nan[2, : V - 12] = True
    negative_nan[3, V // 2:] = True
    x[3, : V // 4] = float("-inf")
    x[4, 1:] = x[4, 0]
    x[4, V // 3] = 1.0
    u = torch.rand(5, generator=torch.Generator().manual_seed(V)).to(dev)
    want, _ = mi.ops.sample_from_logits(x.masked_fill(negative_nan, float("-inf")).to(dev), temperature=0.8, uniform=u)
    y = _with_negative_nan(x, negative_nan).to(dev)
    numbers = (~negative_nan).sum(-1)
    for top_k in (V, V - V // 4, 13):
        got, _, cut = mi.ops.sample_from_logits(y, top_k=top_k, temperature=0.8, uniform=u, return_cut=True)
        rows = ((numbers < top_k) | ((x > float("-inf")).sum(-1) <= top_k) & (top_k == V)).to(dev)
        assert torch.equal(got[rows], want[rows]), top_k
        assert (cut[(numbers < top_k).to(dev)] == float("-inf")).all(), top_k


def test_many_rows_under_capture_leave_the_stream_without_a_workspace(mi, dev):
    """More than 128 rows needed no scratch before they were done in parts, and could be captured as they are.  The scratch of a
    captured call is the graph's: replays, with eager calls and the stream's own workspace growing in between, give the eager
    tokens."""
    R, V = 129, 65544
    gen = torch.Generator(device=dev).manual_seed(9)
    rows = [torch.empty(R, V, device=dev).normal_(0, 3, generator=gen) for _ in range(3)]
    u = torch.rand(R, device=dev, generator=gen)
    want = [mi.ops.sample_from_logits(x, top_p=0.9, uniform=u)[0] for x in rows]
    x = rows[0].clone()
    stream = torch.cuda.Stream()
    before = dict(mi.ops._workspace_sizes)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=stream):
        got, _ = mi.ops.sample_from_logits(x, top_p=0.9, uniform=u)
    assert mi.ops._workspace_sizes == before
    for i in (0, 1, 2, 1):
        x.copy_(rows[i])
        with torch.cuda.stream(stream):
            stream.wait_stream(torch.cuda.current_stream(dev))
            mi.ops.sample_from_logits(rows[2][: 8 << i], top_p=0.9, uniform=u)
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(got, want[i])
