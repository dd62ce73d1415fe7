"""Flash prefill with two heads or one per workgroup (groups that four does not divide), at prompt
lengths around its query blocks."""

import pytest
import torch

pytestmark = pytest.mark.gpu
BF = torch.bfloat16


@pytest.mark.parametrize("Hq,Hkv", [(10, 2), (3, 1), (7, 1), (4, 4), (6, 1), (4, 2)])
@pytest.mark.parametrize("qlens,ctxs", [([1, 31, 33, 64, 127], [0, 5, 70, 0, 1]),
                                        ([128, 129, 255], [0, 63, 0]), ([256, 257, 32], [40, 0, 300])])
@pytest.mark.parametrize("causal,window,chunk", [(True, None, None), (False, None, None),
                                                 (True, 50, None), (True, None, 96)])
def test_flash_prefill_groups(Hq, Hkv, qlens, ctxs, causal, window, chunk):
    from enterprise_inference_amd.ops import attention
    from enterprise_inference_amd.ops import reference as ref
    g = torch.Generator().manual_seed(sum(qlens) + Hq)
    D, bs = 128, 64
    assert attention.prefill_variant(Hq, Hkv, D, bs) == attention.PREFILL_FA
    lens = [a + b for a, b in zip(qlens, ctxs)]
    need = [-(-n // bs) for n in lens]
    bt = torch.zeros(len(lens), max(need), dtype=torch.int32)
    perm, at = torch.randperm(sum(need), generator=g).to(torch.int32), 0
    for s, n in enumerate(need):
        bt[s, :n] = perm[at:at + n]
        at += n
    k = torch.randn(sum(need), Hkv, bs, D, generator=g).to(BF)
    v = torch.randn(sum(need), Hkv, D, bs, generator=g).to(BF)
    q = torch.randn(sum(qlens), Hq, D, generator=g).to(BF)
    sl = torch.tensor(lens, dtype=torch.int32)
    cu = torch.tensor([0] + qlens).cumsum(0).to(torch.int32)
    r = ref.paged_attention_prefill(q.float(), k.float(), v.float(), bt, cu, sl, D ** -0.5, causal,
                                    window, chunk)
    work = torch.tensor(attention.build_prefill_work(
        qlens, attention.prefill_query_block(Hq, Hkv, D, block_size=bs)), dtype=torch.int32)
    d = [t.cuda() for t in (q, k, v, bt, sl, cu, work)]
    # rows of 8 heads' width are the flash form's; a stride of 4 more takes the fallback
    for pad in (0, 4):
        out = torch.empty(sum(qlens), Hq * D + pad, dtype=BF, device="cuda")[:, :Hq * D]
        o = attention.paged_prefill(*d[:6], d[6], work.numel() // 2, D ** -0.5, causal, window, chunk,
                                    out=out.unflatten(1, (Hq, D)))
        # weights and outputs rounded to bf16 (2^-9 each, relative), fp32 sums
        err = (o.double().cpu() - r.double()).norm() / r.double().norm()
        assert err < 4e-3
