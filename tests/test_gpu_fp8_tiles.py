"""GPU parity: the one-stream tile kernel over byte caches, and the quantising append from strided rows, at the sizes
where their loops change."""
import pytest
import torch

from oracle import paged_attention as oa

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "fp16"])
@pytest.mark.parametrize("split", [-1, 3])
@pytest.mark.parametrize("d,Hq,Hkv", [(64, 32, 8), (64, 8, 8), (128, 32, 8), (128, 16, 1)])
def test_fp8_tiles(mi, dev, d, Hq, Hkv, split, dtype):
    """Row and key counts around tiles (64 keys), workgroups (128 or 256 rows) and chunks; scales that jump between the
    chunks of a request by up to five decades."""
    chunk = 64
    q_lens = [1, 2, 33, 63, 64, 65, 129, 200, 300]
    ctx = [0, 62, 31, 0, 64, 127, 0, 333, 1]
    kv_lens = torch.tensor([a + b for a, b in zip(q_lens, ctx)], dtype=torch.int32)
    cu_q = torch.zeros(len(q_lens) + 1, dtype=torch.int32)
    cu_q[1:] = torch.cumsum(torch.tensor(q_lens), 0)
    gen = torch.Generator().manual_seed(d + Hq)
    bt, N = mi.synthetic.build_block_table(kv_lens, chunk, gen)
    q = torch.randn(int(cu_q[-1]), Hq, d, generator=gen).to(dtype).to(dev)
    mag = torch.tensor([1e-5, 0.05, 1.0])[torch.randint(0, 3, (2, N, 1, Hkv, 1), generator=gen)]
    k8, ks = oa.quantize_chunks_fp8((torch.randn(N, chunk, Hkv, d, generator=gen) * mag[0]).to(dtype))
    v8, vs = oa.quantize_chunks_fp8((torch.randn(N, chunk, Hkv, d, generator=gen) * mag[1]).to(dtype))
    with mi.ops.tuning(prefill_kv_split=split):
        out = mi.ops.paged_prefill_attention(q, k8.to(dev), v8.to(dev), cu_q.to(dev), kv_lens.to(dev), bt.to(dev),
                                             k_scales=ks.to(dev), v_scales=vs.to(dev))
    ref = oa.paged_varlen_attention(q.cpu(), k8, v8, cu_q, kv_lens, bt, k_scales=ks, v_scales=vs)
    err = (out.float().cpu() - ref).abs()
    assert (err <= 2e-2 + 2e-2 * ref.abs()).all(), f"max err {err.max().item():.4e}"


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "fp16"])
@pytest.mark.parametrize("bound", [128, 100000])   # (width 128: workgroups of four wavefronts, of eight)
@pytest.mark.parametrize("d", [64, 128])
def test_value_scales_of_every_kind(mi, dev, d, bound, dtype):
    """Value scales below and above what an exact conversion takes, negative, zero, NaN and infinite ones, one to a KV head.  A finite
    scale: the oracle's result, up to roundings of the probabilities and of the products of value and scale (each 2^-9 or
    2^-12 of the largest, the products no finer than the type's: 2^-25, and 2^-126 for what bf16 may flush; doubled for sums).  NaN: NaN.  Infinite: not finite."""
    f16 = dtype == torch.float16
    finite = [1.0, 0.37, -0.7, 0.0, 1.9 * 2.0**-19, 1.3 * 2.0**-16, 300.0 if f16 else 1.7e30, 1.5 * 2.0**-120 if f16 else 1.1 * 2.0**120]
    scales = torch.tensor(finite + [float("nan"), float("inf")])
    Hkv, chunk, Hq = len(scales), 64, 2 * len(scales)
    q_lens = [70, 128, 1, 33]
    kv_lens = torch.tensor(q_lens, dtype=torch.int32)
    cu_q = torch.tensor([0] + q_lens, dtype=torch.int32).cumsum(0).to(torch.int32)
    gen = torch.Generator().manual_seed(d)
    bt, N = mi.synthetic.build_block_table(kv_lens, chunk, gen)
    q = torch.randn(int(cu_q[-1]), Hq, d, generator=gen).to(dtype)
    k8 = torch.randint(0, 56, (N, chunk, Hkv, d), generator=gen, dtype=torch.uint8)          # up to 1
    v8 = torch.randint(0, 105, (N, chunk, Hkv, d), generator=gen, dtype=torch.uint8)         # up to 64
    v8 |= torch.randint(0, 2, v8.shape, generator=gen, dtype=torch.uint8) << 7
    ks, vs = torch.full((N, Hkv), 0.5), scales.expand(N, Hkv).contiguous()
    with mi.ops.tuning(prefill_kv_split=-1):
        out = mi.ops.paged_prefill_attention(q.to(dev), k8.to(dev), v8.to(dev), cu_q.to(dev), kv_lens.to(dev), bt.to(dev),
                                             k_scales=ks.to(dev), v_scales=vs.to(dev), max_kv_len=bound, one_row_requests=False)
    out = out.float().cpu().view(-1, Hkv, 2, d)
    n = len(finite)
    ref = oa.paged_varlen_attention(q, k8, v8, cu_q, kv_lens, bt, k_scales=ks,
                                    v_scales=vs.masked_fill(~torch.isfinite(vs), 1.0)).view(-1, Hkv, 2, d)
    unit, least = (2.0**-12, 2.0**-25) if f16 else (2.0**-9, 2.0**-126)
    for h, scale in enumerate(finite):
        bar = 4 * unit * 64 * abs(scale) + 2 * least + (2.0**-119 if scale == 0 else 0)   # (zero may count as 2^-126)
        err = (out[:, h] - ref[:, h]).abs().max().item()
        assert err <= bar, (scale, err, bar)
    assert out[:, n].isnan().all() and not out[:, n + 1].isfinite().any()
    # a prompt's first row is its first value: rounded as a product and as a result (2^-25 each where fp16 is subnormal), and as a
    # probability or a quotient (2 units each)
    first = cu_q[:-1].long()
    value = v8.view(torch.float8_e4m3fn).float()[bt[:, 0].long(), 0, :n] * scales[:n, None]
    err = (out[first, :n, 0] - value).abs()
    assert (err <= least * 2.001 + 6 * unit * value.abs()).all(), err.max().item()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "fp16"])
@pytest.mark.parametrize("d,chunk", [(128, 256), (64, 128), (96, 64), (128, 320)])
def test_fp8_append_from_strided_rows(mi, dev, d, chunk, dtype):
    """Values read from a wider row; runs of one token, of two, across workgroups' slices, of whole chunks and of a chunk
    that does not fit a workgroup's registers; scales beyond the range of the quick quotient; padded rows."""
    Hkv, N = 3, 24
    gen = torch.Generator().manual_seed(d + chunk)
    reqs = [(0, chunk, [3]), (0, 2 * chunk + 17, [7, 1, 12]), (chunk - 5, 60, [5, 9]), (chunk, 2, [2, 14]), (0, 1, [20]),
            (chunk - 1, 2, [6, 8]), (0, 2, [10]), (0, 31, [11])]
    slots = [(chunks[pos // chunk], pos % chunk) for first, n, chunks in reqs for pos in range(first, first + n)]
    real = len(slots)
    slots += [(N - 1, 0)] * 40
    T = len(slots)
    tc, tl = (torch.tensor(x) for x in zip(*slots))
    key = (torch.randn(T, Hkv, d, generator=gen) * 3).to(dtype)
    wide = torch.randn(T, Hkv, 3 * d, generator=gen).to(dtype)
    val = wide[:, :, 2 * d:]
    key[chunk + 3, 1] = 0
    val[real - 31:real] *= 1e-4
    if dtype == torch.bfloat16:
        key[real - 31:real, 2] *= 1e-30
        val[0:chunk, 0] *= 1e30
    k8 = torch.randint(0, 255, (N, chunk, Hkv, d), generator=gen, dtype=torch.uint8)
    v8 = torch.randint(0, 255, (N, chunk, Hkv, d), generator=gen, dtype=torch.uint8)
    ks, vs = torch.rand(N, Hkv, generator=gen) + 0.5, torch.rand(N, Hkv, generator=gen) * 1e-3
    k8d, v8d, ksd, vsd = k8.to(dev), v8.to(dev), ks.to(dev), vs.to(dev)
    mi.ops.kv_append_fp8(key.to(dev), wide.to(dev)[:, :, 2 * d:], k8d, v8d, ksd, vsd, tc.to(dev), tl.to(dev), headroom=1.5)
    for cache, scales, rows, got_c, got_s in ((k8, ks, key, k8d, ksd), (v8, vs, val, v8d, vsd)):
        oa.kv_append_fp8(cache, scales, rows[:real], tc[:real], tl[:real], headroom=1.5)
        assert torch.equal(got_s.cpu()[:N - 1], scales[:N - 1])
        assert torch.equal(got_c.cpu()[:N - 1], cache[:N - 1])
