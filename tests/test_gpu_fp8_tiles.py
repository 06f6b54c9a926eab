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
