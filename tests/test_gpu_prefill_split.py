"""GPU parity: automatic key ranges and their merge, with and without the decode launches of one-row requests."""
import pytest
import torch

from oracle import paged_attention as oa

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("one_row_requests", [True, False])
@pytest.mark.parametrize("d,Hq,Hkv", [(128, 32, 8), (64, 8, 8), (96, 24, 8), (256, 4, 1)])
def test_few_rows_over_contexts(mi, dev, d, Hq, Hkv, one_row_requests):
    """Few rows over a context of more than two ranges; a one-row request among them; padded rows behind."""
    q_lens, ctx, chunk, pad = [3, 1, 65, 2], [0, 1500, 700, 2100], 64, 5
    kv_lens = torch.tensor([a + b for a, b in zip(q_lens, ctx)], dtype=torch.int32)
    cu_q = torch.zeros(len(q_lens) + 1, dtype=torch.int32)
    cu_q[1:] = torch.cumsum(torch.tensor(q_lens), 0)
    gen = torch.Generator().manual_seed(d)
    bt, N = mi.synthetic.build_block_table(kv_lens, chunk, gen)
    T = int(cu_q[-1])
    q = torch.randn(T + pad, Hq, d, generator=gen).bfloat16()
    kc, vc = (torch.randn(N, chunk, Hkv, d, generator=gen).bfloat16() for _ in range(2))
    out = mi.ops.paged_prefill_attention(q.to(dev), kc.to(dev), vc.to(dev), cu_q.to(dev), kv_lens.to(dev), bt.to(dev),
                                         max_kv_len=int(kv_lens.max()), one_row_requests=one_row_requests).float().cpu()
    ref = oa.paged_varlen_attention(q[:T], kc, vc, cu_q, kv_lens, bt)
    assert (out[:T] - ref).abs().max().item() < 2e-2
    assert not out[T:].any()


@pytest.mark.parametrize("d,Hq,Hkv", [(128, 8, 8), (64, 8, 8), (64, 32, 8), (192, 8, 2)])
@pytest.mark.parametrize("q_lens", [[64], [40, 0, 0], [1, 65, 0, 16, 17], [0] * 127 + [3], [0, 5] * 65])
def test_every_query_block_has_a_workgroup(mi, dev, d, Hq, Hkv, q_lens):
    """As many blocks as a launch of these rows and requests can have: requests of whole blocks and of one row, requests
    without rows, both forms of numbering (up to 128 requests and more), with and without key ranges."""
    chunk, kv_lens = 64, torch.tensor([n + 200 if n else 0 for n in q_lens], dtype=torch.int32)
    cu_q = torch.zeros(len(q_lens) + 1, dtype=torch.int32)
    cu_q[1:] = torch.cumsum(torch.tensor(q_lens), 0)
    gen = torch.Generator().manual_seed(d + len(q_lens))
    bt, N = mi.synthetic.build_block_table(kv_lens.clamp(min=1), chunk, gen)
    T = int(cu_q[-1])
    q = torch.randn(T, Hq, d, generator=gen).bfloat16()
    kc, vc = (torch.randn(N, chunk, Hkv, d, generator=gen).bfloat16() for _ in range(2))
    ref = oa.paged_varlen_attention(q, kc, vc, cu_q, kv_lens, bt)
    for split in (-1, 2):
        with mi.ops.tuning(prefill_kv_split=split):
            out = mi.ops.paged_prefill_attention(q.to(dev), kc.to(dev), vc.to(dev), cu_q.to(dev), kv_lens.to(dev), bt.to(dev),
                                                 max_kv_len=int(kv_lens.max()), one_row_requests=False).float().cpu()
        assert (out - ref).abs().max().item() < 2e-2


@pytest.mark.parametrize("fp8", [False, True])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "fp16"])
@pytest.mark.parametrize("Hq,Hkv", [(32, 8), (8, 8), (16, 1), (40, 2)])
def test_four_wavefronts_give_what_eight_do(mi, dev, Hq, Hkv, dtype, fp8):
    """A row's walk over the tiles does not depend on the rows that share its workgroup: the same bits with the bound of the
    keys that chooses four wavefronts and with one that chooses eight.  Requests around a tile, a block and two tiles, with and
    without a context, values whose scale differs from chunk to chunk."""
    q_lens, ctx, chunk, d = [1, 63, 64, 65, 33, 128, 200, 7, 700], [0, 0, 0, 0, 300, 63, 1, 130, 0], 64, 128
    kv_lens = torch.tensor([a + b for a, b in zip(q_lens, ctx)], dtype=torch.int32)
    cu_q = torch.zeros(len(q_lens) + 1, dtype=torch.int32)
    cu_q[1:] = torch.cumsum(torch.tensor(q_lens), 0)
    gen = torch.Generator().manual_seed(Hq)
    bt, N = mi.synthetic.build_block_table(kv_lens, chunk, gen)
    T = int(cu_q[-1])
    q = torch.randn(T, Hq, d, generator=gen).to(dtype)
    kc, vc = ((torch.randn(N, chunk, Hkv, d, generator=gen) * (0.05 + 4 * torch.rand(N, 1, 1, 1, generator=gen))).to(dtype) for _ in range(2))
    kw, ref_kw, caches = {}, {}, [kc.to(dev), vc.to(dev)]
    if fp8:
        pools = [torch.empty(kc.shape, dtype=torch.uint8, device=dev) for _ in range(2)]
        scales = [torch.empty(N, Hkv, dtype=torch.float32, device=dev) for _ in range(2)]
        for src, pool, scale in zip(caches, pools, scales):
            mi.ops.quantize_chunks_fp8(src, pool, scale)
        caches, kw = pools, dict(k_scales=scales[0], v_scales=scales[1])
        ref_kw = {k: v.cpu() for k, v in kw.items()}
    out = [mi.ops.paged_prefill_attention(q.to(dev), *caches, cu_q.to(dev), kv_lens.to(dev), bt.to(dev), max_kv_len=most,
                                          one_row_requests=False, **kw) for most in (int(kv_lens.max()), 100000)]
    with mi.ops.tuning(prefill_kv_split=-1):
        eight = mi.ops.paged_prefill_attention(q.to(dev), *caches, cu_q.to(dev), kv_lens.to(dev), bt.to(dev), max_kv_len=100000,
                                               one_row_requests=False, **kw)
    assert torch.equal(out[0], eight)
    ref = oa.paged_varlen_attention(q, caches[0].cpu(), caches[1].cpu(), cu_q, kv_lens, bt, **ref_kw)
    bound = 2e-2 + 2e-2 * ref.abs()
    for o in out:
        assert ((o.float().cpu() - ref).abs() <= bound).all()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "fp16"])
@pytest.mark.parametrize("splits", [-1, 3])
def test_a_call_of_few_workgroups_gives_what_a_large_one_does(mi, dev, dtype, splits):
    """Prompts of width 64 over an fp8 cache: a call of at most three workgroups per CU takes another build of the kernel than
    a larger one.  The same requests alone and as the first of many: the same bits, and those of the reference."""
    lens, chunk, d, Hq, Hkv = [1, 33, 64, 65, 190, 257], 64, 64, 32, 8
    gen = torch.Generator().manual_seed(5)
    cus = torch.cuda.get_device_properties(dev).multi_processor_count
    copies = 2 + 3 * cus // (Hkv * sum(-(-n // 32) for n in lens))   # (a block is 128 rows, 32 tokens here)
    kv_lens = torch.tensor(lens, dtype=torch.int32)
    bt, N = mi.synthetic.build_block_table(kv_lens, chunk, gen)
    T = sum(lens)
    q = torch.randn(T, Hq, d, generator=gen).to(dtype).to(dev)
    src = [(torch.randn(N, chunk, Hkv, d, generator=gen) * (0.05 + 4 * torch.rand(N, 1, 1, 1, generator=gen))).to(dtype).to(dev) for _ in range(2)]
    pools = [torch.empty(x.shape, dtype=torch.uint8, device=dev) for x in src]
    scales = [torch.empty(N, Hkv, dtype=torch.float32, device=dev) for _ in range(2)]
    for x, pool, scale in zip(src, pools, scales):
        mi.ops.quantize_chunks_fp8(x, pool, scale)
    out = []
    for n in (1, copies):
        kl = kv_lens.repeat(n)
        cu_q = torch.zeros(kl.numel() + 1, dtype=torch.int32)
        cu_q[1:] = torch.cumsum(kl, 0)
        with mi.ops.tuning(prefill_kv_split=splits):
            out.append(mi.ops.paged_prefill_attention(q.repeat(n, 1, 1), *pools, cu_q.to(dev), kl.to(dev), bt.repeat(n, 1).to(dev),
                                                      max_kv_len=int(kl.max()), one_row_requests=False, k_scales=scales[0],
                                                      v_scales=scales[1]))
    assert torch.equal(out[0], out[1][:T])
    cu_q = torch.zeros(len(lens) + 1, dtype=torch.int32)
    cu_q[1:] = torch.cumsum(kv_lens, 0)
    ref = oa.paged_varlen_attention(q.cpu(), pools[0].cpu(), pools[1].cpu(), cu_q, kv_lens, bt, k_scales=scales[0].cpu(), v_scales=scales[1].cpu())
    assert ((out[0].float().cpu() - ref).abs() <= 2e-2 + 2e-2 * ref.abs()).all()
