"""The MFMA grouped expert GEMM: K steps around the length of its LDS ring, slices around its row
tiles, and the sizes at which fused_moe turns to it."""

import pytest
import torch

pytestmark = pytest.mark.gpu
BF = torch.bfloat16


@pytest.mark.parametrize("form", [0, 1, 2])
@pytest.mark.parametrize("K", [64, 128, 192, 320, 640])
@pytest.mark.parametrize("counts", [[1, 0, 127, 128, 129, 65], [0] * 65 + [200, 0, 3]])
def test_grouped_gemm(counts, K, form):
    from enterprise_inference_amd._native import kernels as lib
    from enterprise_inference_amd.ops._dispatch import ptr, stream
    g = torch.Generator().manual_seed(K + form)
    E, n, N = len(counts), sum(counts), 384
    X = torch.randn(300, K, generator=g).to("cuda", BF)
    row_idx = torch.randint(0, 300, (n,), generator=g).to("cuda", torch.int32)
    offs = torch.tensor([0] + counts).cumsum(0).to("cuda", torch.int32)
    W = (torch.randn(E, N, K, generator=g) * K ** -0.5).to("cuda", BF)
    out = torch.full((n, N // 2 if form == 1 else N), float("nan"), device="cuda", dtype=BF)
    assert lib().eia_moe_grouped_gemm(ptr(X), X.stride(0), ptr(row_idx), ptr(W), N, K, E, ptr(offs),
                                      n, form, ptr(out), out.stride(0), stream(X)) == 0
    xs = X.double()[row_idx.long()]
    for e, (a, b) in enumerate(zip(offs.tolist(), offs.tolist()[1:])):
        y = xs[a:b] @ W[e].double().t()
        if form == 1:
            y = torch.nn.functional.silu(y[:, :N // 2]) * y[:, N // 2:]
        elif form == 2:
            y = torch.relu(y) ** 2
        # fp32 sums of K exact products, one bf16 rounding (2^-9) and a fast exponential
        assert a == b or ((out[a:b].double() - y).norm() / y.norm()) < 3e-3


# (mean rows per expert of 16: 256 takes tiles of up to 320 x 128, 360 of up to 256 x 256)
@pytest.mark.parametrize("form", [0, 1])
@pytest.mark.parametrize("K", [64, 128, 192, 448])
@pytest.mark.parametrize("counts", [
    [1, 63, 64, 65, 319, 320, 321, 129, 193, 640, 641, 0, 256, 511, 130, 443],
    [1, 64, 255, 256, 257, 511, 512, 513, 129, 193, 769, 0, 321, 383, 640, 956]])
def test_grouped_gemm_large_tiles(counts, K, form):
    from enterprise_inference_amd._native import kernels as lib
    from enterprise_inference_amd.ops._dispatch import ptr, stream
    assert sum(counts) in (16 * 256, 16 * 360)
    g = torch.Generator().manual_seed(K + form)
    E, n, N = len(counts), sum(counts), 2048
    X = torch.randn(700, K, generator=g).to("cuda", BF)
    row_idx = torch.randint(0, 700, (n,), generator=g).to("cuda", torch.int32)
    offs = torch.tensor([0] + counts).cumsum(0).to("cuda", torch.int32)
    W = (torch.randn(E, N, K, generator=g) * K ** -0.5).to("cuda", BF)
    out = torch.full((n + 1, N // 2 if form == 1 else N), float("nan"), device="cuda", dtype=BF)
    assert lib().eia_moe_grouped_gemm(ptr(X), X.stride(0), ptr(row_idx), ptr(W), N, K, E, ptr(offs),
                                      n, form, ptr(out), out.stride(0), stream(X)) == 0
    xs = X.double()[row_idx.long()]
    for e, (a, b) in enumerate(zip(offs.tolist(), offs.tolist()[1:])):
        y = xs[a:b] @ W[e].double().t()
        if form == 1:
            y = torch.nn.functional.silu(y[:, :N // 2]) * y[:, N // 2:]
        # fp32 sums of K exact products, one bf16 rounding (2^-9) and a fast exponential
        assert a == b or ((out[a:b].double() - y).norm() / y.norm()) < 3e-3
    assert out[n:].isnan().all()


@pytest.mark.parametrize("form", [0, 1, 2])
@pytest.mark.parametrize("K,N", [(2048, 256), (2112, 256), (4096, 256), (128, 8192), (64, 7936), (64, 8448)])
@pytest.mark.parametrize("counts", [[1, 64, 65, 128, 129, 192, 193, 0], [130, 191, 127, 63, 66, 256, 1, 190],
                                    [100, 101, 99, 98, 97, 129, 102, 104]])
def test_grouped_gemm_few_rows_of_long_experts(counts, K, N, form):
    """Up to 128 rows an expert (a step's accesses in front of its products), slices of one to five units; and
    launches of 496, 512 and 528 tiles of 128 x 128, of which the first two leave wide tiles out at 104 rows."""
    from enterprise_inference_amd._native import kernels as lib
    from enterprise_inference_amd.ops._dispatch import ptr, stream
    g = torch.Generator().manual_seed(K + form)
    E, n = len(counts), sum(counts)
    assert n <= 128 * E
    X = torch.randn(300, K, generator=g).to("cuda", BF)
    row_idx = torch.randint(0, 300, (n,), generator=g).to("cuda", torch.int32)
    offs = torch.tensor([0] + counts).cumsum(0).to("cuda", torch.int32)
    W = (torch.randn(E, N, K, generator=g) * K ** -0.5).to("cuda", BF)
    out = torch.full((n + 1, N // 2 if form == 1 else N), float("nan"), device="cuda", dtype=BF)
    assert lib().eia_moe_grouped_gemm(ptr(X), X.stride(0), ptr(row_idx), ptr(W), N, K, E, ptr(offs),
                                      n, form, ptr(out), out.stride(0), stream(X)) == 0
    xs = X.double()[row_idx.long()]
    for e, (a, b) in enumerate(zip(offs.tolist(), offs.tolist()[1:])):
        y = xs[a:b] @ W[e].double().t()
        if form == 1:
            y = torch.nn.functional.silu(y[:, :N // 2]) * y[:, N // 2:]
        elif form == 2:
            y = torch.relu(y) ** 2
        # fp32 sums of K exact products, one bf16 rounding (2^-9) and a fast exponential
        assert a == b or ((out[a:b].double() - y).norm() / y.norm()) < 3e-3
    assert out[n:].isnan().all()


@pytest.mark.parametrize("T,E,H,I", [(100, 4, 512, 256), (96, 4, 512, 256), (200, 16, 1024, 1024),
                                     (600, 4, 512, 4352)])
@pytest.mark.parametrize("shift", [0, 4])
def test_fused_moe_rows_per_expert(T, E, H, I, shift):
    from enterprise_inference_amd.ops import moe
    from enterprise_inference_amd.ops import reference as ref
    g = torch.Generator().manual_seed(T)
    x = torch.randn(T * H + shift, generator=g).to(BF)[shift:].view(T, H)
    w13 = (torch.randn(E, 2 * I, H, generator=g) * H ** -0.5).to(BF)
    w2 = (torch.randn(E, H, I, generator=g) * I ** -0.5).to(BF)
    w, ids = torch.topk(torch.softmax(torch.randn(T, E, generator=g), -1), 2, -1)
    ids = ids.to(torch.int32)
    xd = torch.empty(T * H + shift, dtype=BF, device="cuda")[shift:].view(T, H).copy_(x)
    out = moe.fused_moe(xd, *(t.cuda() for t in (w13, w2, w, ids))).double().cpu()
    r = ref.fused_moe(x, w13, w2, w, ids).double()
    # hidden rows, expert outputs and sums are rounded to bf16 on both sides: 3 x 1.7e-3 each
    assert (out - r).norm() / r.norm() < 1.1e-2


@pytest.mark.parametrize("T", [200, 480])
@pytest.mark.parametrize("act", ["silu", "relu2"])
def test_moved_weights_are_not_copied(act, T):
    """Expert stacks that do not begin on 16 bytes: the result, without a second copy of them."""
    from enterprise_inference_amd.ops import moe
    from enterprise_inference_amd.ops import reference as ref
    g = torch.Generator().manual_seed(T)
    E, H, I = 8, 1024, 2048
    x = torch.randn(T, H, generator=g).to(BF)
    up = 2 * I if act == "silu" else I
    w13 = (torch.randn(E, up, H, generator=g) * H ** -0.5).to(BF)
    w2 = (torch.randn(E, H, I, generator=g) * I ** -0.5).to(BF)
    w, ids = torch.topk(torch.softmax(torch.randn(T, E, generator=g), -1), 2, -1)
    ids = ids.to(torch.int32)
    odd = lambda t: torch.empty(t.numel() + 1, dtype=BF, device="cuda")[1:].view(t.shape).copy_(t)
    a = [x.cuda(), odd(w13), odd(w2), w.cuda(), ids.cuda()]
    f = moe.fused_moe if act == "silu" else moe.ungated_moe
    out = f(*a)
    torch.cuda.synchronize()
    torch.cuda.reset_peak_memory_stats()
    before = torch.cuda.memory_allocated()
    f(*a)
    # (the stacks are 32 and, with gates, 64 MB; the rows' intermediates stay under 12)
    assert torch.cuda.max_memory_allocated() - before < 16 << 20
    r = (ref if act == "silu" else moe).__dict__["fused_moe" if act == "silu" else "ungated_moe"](
        x, w13, w2, w, ids).double()
    # hidden rows, expert outputs and sums are rounded to bf16 on both sides: 3 x 1.7e-3 each
    assert (out.double().cpu() - r).norm() / r.norm() < 1.1e-2


@pytest.mark.parametrize("n,E,lo,hi,k", [(1, 1, 0, 1, 1), (1023, 8, 0, 8, 3), (1025, 5, 2, 3, 2),
                                         (4096, 256, 0, 256, 2), (4097, 255, 3, 250, 1),
                                         (8192, 16, 0, 16, 4), (8195, 256, 250, 256, 5)])
def test_align_sorts_entries_by_expert(n, E, lo, hi, k):
    from enterprise_inference_amd._native import kernels as lib
    from enterprise_inference_amd.ops._dispatch import ptr, stream
    g = torch.Generator().manual_seed(n + E)
    ids = torch.randint(0, E + 1, (n,), generator=g).to("cuda", torch.int32)   # E: no expert
    offs = torch.full((hi - lo + 1,), -7, device="cuda", dtype=torch.int32)
    row_idx, inv = (torch.full((n,), -7, device="cuda", dtype=torch.int32) for _ in range(2))
    assert lib().eia_moe_align(ptr(ids), n, E, lo, hi, ptr(offs), ptr(row_idx), ptr(inv), k,
                               stream(ids)) == 0
    ids, offs, row_idx, inv = (t.tolist() for t in (ids, offs, row_idx, inv))
    here = [i for i in range(n) if lo <= ids[i] < hi]
    want = [0]
    for e in range(lo, hi):
        want.append(want[-1] + ids.count(e))
    assert offs == want and sorted(inv[i] for i in here) == list(range(len(here)))
    for i in range(n):
        if lo <= ids[i] < hi:
            assert offs[ids[i] - lo] <= inv[i] < offs[ids[i] - lo + 1] and row_idx[inv[i]] == i // k
        else:
            assert inv[i] == -1
    assert row_idx[len(here):] == [0] * (n - len(here))


@pytest.mark.parametrize("sk", [0, 1, 2, 3, 4])             # 0: the bf16 rows of an unsplit product
@pytest.mark.parametrize("T,k,H", [(1, 1, 8), (3, 2, 1032), (5, 3, 2056), (2, 5, 4096), (70, 8, 1024)])
def test_combine(T, k, H, sk):
    from enterprise_inference_amd._native import kernels as lib
    from enterprise_inference_amd.ops._dispatch import ptr, stream
    g = torch.Generator().manual_seed(T + H + sk)
    n = T * k
    w = torch.rand(T, k, generator=g).to("cuda")
    inv = torch.randperm(n, generator=g).to("cuda", torch.int32)
    inv[torch.rand(n, generator=g).to("cuda") < 0.2] = -1          # another rank's expert
    out = torch.full((T, H + 8), float("nan"), device="cuda", dtype=BF)
    if sk:
        part = torch.randn(sk, n, H, generator=g).to("cuda")
        rows = part[0].clone()
        for j in range(1, sk):
            rows += part[j]
        rows = rows.to(BF)
        rc = lib().eia_moe_combine_sk(ptr(part), sk, n, ptr(w), ptr(inv), T, k, H, ptr(out),
                                      out.stride(0), stream(out))
    else:
        rows = torch.randn(n, H, generator=g).to("cuda", BF)
        rc = lib().eia_moe_combine(ptr(rows), rows.stride(0), ptr(w), ptr(inv), T, k, H, ptr(out),
                                   out.stride(0), stream(out))
    assert rc == 0
    terms = rows.double()[inv.long().clamp(min=0)].view(T, k, H) * w.double()[:, :, None]
    terms[(inv < 0).view(T, k)] = 0
    # k fp32 products and sums, then one rounding to bf16
    bound = terms.abs().sum(1) * (k * 2.0 ** -23) + terms.sum(1).abs() * 2.0 ** -8
    assert ((out[:, :H].double() - terms.sum(1)).abs() <= bound).all()
    assert out[:, H:].isnan().all()
