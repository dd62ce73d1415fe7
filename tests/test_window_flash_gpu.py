"""The LDS-shared prefill form of window attention against the op's own plain CPU path: group sizes,
padded head sizes, windows and kept tokens on both sides of a 64-key tile, prompts that continue."""

import pytest
import torch

pytestmark = pytest.mark.gpu


def _spec(wa, kind, H, G, D, Dv, window, dev):
    g = torch.Generator().manual_seed(3)
    P = 2 if kind == "pair" else 1
    s = wa.WindowSpec(H, G, P, D, Dv, window, 0, mult=torch.linspace(0.5, 1.5, H * P) * D ** -0.5)
    if kind == "cap":
        s.cap, s.sink, s.post = 5.0, torch.randn(H, generator=g), 0.8
    elif kind == "sigmoid":
        s.weights, s.bias = 1, torch.randn(H, generator=g) - 3.0
    elif kind == "pair":
        s.keep, s.epilogue, s.eps, s.post, s.lam = 70, 1, 1e-5, 0.7, torch.tensor([0.4])
    elif kind == "keep":
        s.keep = 4
    for f in ("mult", "sink", "bias", "lam"):
        t = getattr(s, f)
        if t is not None:
            setattr(s, f, t.to(dev))
    return s


def _pages(g, total, bs):
    """Random pages for sequences of ``total`` tokens: block tables and the page count."""
    pages = [max(1, -(-n // bs)) for n in total]
    order = torch.randperm(sum(pages), generator=g).to(torch.int32)
    bt = torch.zeros(len(total), max(pages), dtype=torch.int32)
    at = 0
    for s, n in enumerate(pages):
        bt[s, :n] = order[at:at + n]
        at += n
    return bt, sum(pages)


@pytest.mark.parametrize("kind", ["plain", "cap", "sigmoid", "pair", "keep"])
@pytest.mark.parametrize("H,G,D,Dv,bs", [(4, 1, 128, 128, 64), (6, 3, 72, 48, 128), (3, 1, 64, 64, 64),
                                         (8, 2, 96, 96, 64), (2, 2, 64, 112, 64)])
@pytest.mark.parametrize("window,new,past", [(0, [1, 200, 33, 65], [0, 0, 190, 63]),
                                             (50, [1, 200, 33, 65], [0, 0, 190, 63]),
                                             (130, [1, 200, 33, 65], [0, 0, 190, 63]),
                                             (0, [40, 7], [1000, 130])])
def test_window_flash(window, new, past, H, G, D, Dv, bs, kind):
    from enterprise_inference_amd.ops import attention as A
    from enterprise_inference_amd.ops import window_attention as wa
    if kind == "pair":
        D = 64 if D > 64 else 40
    g = torch.Generator().manual_seed(H + D + window)
    P = 2 if kind == "pair" else 1
    pages = [-(-(a + b) // bs) for a, b in zip(new, past)]
    order = torch.randperm(sum(pages), generator=g).to(torch.int32)
    bt = torch.zeros(len(new), max(pages), dtype=torch.int32)
    at = 0
    for s, n in enumerate(pages):
        bt[s, :n] = order[at:at + n]
        at += n
    cu = torch.tensor([0] + new).cumsum(0).to(torch.int32)
    pos = torch.cat([torch.arange(n) + f for n, f in zip(new, past)]).to(torch.int32)
    T = int(cu[-1])
    bf = torch.bfloat16
    rnd = lambda *s: torch.randn(*s, generator=g).to(bf)
    q, k, v = rnd(T, H * P * D), rnd(sum(pages), bs, G * P * D), rnd(sum(pages), G * Dv, bs)
    for s, (a, b) in enumerate(zip(new, past)):              # slots behind a sequence hold anything
        last, used = int(bt[s, pages[s] - 1]), (a + b - 1) % bs + 1
        k[last, used:] = float("nan")
        v[last, :, used:] = float("nan")
    gate = None if kind == "pair" else rnd(T, H if kind == "cap" else H * Dv)

    def run(dev):
        md = A.AttentionMetadata(
            num_decode=0, num_prefill_tokens=T, slot_mapping=pos.to(dev), positions=pos.to(dev),
            prefill_block_tables=bt.to(dev), prefill_cu_q=cu.to(dev), prefill_q_lens=new)
        spec = _spec(wa, kind, H, G, D, Dv, window, dev)
        spec.gate_heads = kind == "cap"
        if dev == "cuda":
            qb = wa.query_block(spec, bf, bs)
            assert qb == 128 // {1: 1, 2: 2, 3: 1, 4: 4}[H // G]
            n = sum(-(-a // qb) for a in new)           # (the long context is cut into parts)
            parts = (wa.pair_parts(n, spec, qb, bt.shape[1] * bs) if P == 2 else
                     wa.flash_parts(n, spec, qb, max(new), bt.shape[1] * bs))
            assert (parts[0] > 1) == (max(past) > 900)
        return wa.window_attention(q.to(dev), k.to(dev), v.to(dev), md, spec,
                                   None if gate is None else gate.to(dev)).cpu()

    a, b = run("cpu").double(), run("cuda").double()
    # both sides sum in fp32 and round once to bf16 (2^-9): neighbouring roundings at most
    assert float((a - b).norm() / a.norm()) < 4e-3
    assert float(((a - b).abs() / (a.abs() + 0.05 * a.abs().mean())).max()) < 2 ** -6


@pytest.mark.parametrize("kind", ["plain", "cap", "sigmoid", "pair", "keep"])
@pytest.mark.parametrize("H,G,D,Dv,bs", [(4, 1, 128, 128, 64), (6, 2, 72, 48, 32), (16, 1, 64, 64, 64),
                                         (3, 3, 96, 96, 64), (10, 2, 64, 112, 128)])
@pytest.mark.parametrize("window", [0, 50, 600])
@pytest.mark.parametrize("parts", [1, 3, 16])
def test_window_decode(parts, window, H, G, D, Dv, bs, kind, monkeypatch):
    from enterprise_inference_amd.ops import attention as A
    from enterprise_inference_amd.ops import window_attention as wa
    monkeypatch.setenv("EIA_WINDOW_DECODE_P", str(parts))
    if kind == "pair":
        D = 64 if D > 64 else 40
    g = torch.Generator().manual_seed(H + D + window)
    P = 2 if kind == "pair" else 1
    lens = [1, 32, 33, 0, 257, 700]                          # (0: a padding row)
    pages = [max(1, -(-n // bs)) for n in lens]
    order = torch.randperm(sum(pages), generator=g).to(torch.int32)
    bt = torch.zeros(len(lens), max(pages), dtype=torch.int32)
    at = 0
    for s, n in enumerate(pages):
        bt[s, :n] = order[at:at + n]
        at += n
    pos = torch.tensor([max(0, n - 1) for n in lens], dtype=torch.int32)
    bf, T = torch.bfloat16, len(lens)
    rnd = lambda *s: torch.randn(*s, generator=g).to(bf)
    q, k, v = rnd(T, H * P * D), rnd(sum(pages), bs, G * P * D), rnd(sum(pages), G * Dv, bs)
    gate = None if kind == "pair" else rnd(T, H if kind == "cap" else H * Dv)

    def run(dev):
        md = A.AttentionMetadata(
            num_decode=T, num_prefill_tokens=0, slot_mapping=pos.to(dev), positions=pos.to(dev),
            decode_block_tables=bt.to(dev),
            decode_seq_lens=torch.tensor(lens, dtype=torch.int32, device=dev))
        spec = _spec(wa, kind, H, G, D, Dv, window, dev)
        spec.gate_heads = kind == "cap"
        return wa.window_attention(q.to(dev), k.to(dev), v.to(dev), md, spec,
                                   None if gate is None else gate.to(dev)).cpu()

    a, b = run("cpu").double(), run("cuda").double()
    live = torch.tensor(lens) > 0
    assert float((a - b)[live].norm() / a[live].norm()) < 4e-3   # as above


@pytest.mark.parametrize("sink", [float("-inf"), torch.finfo(torch.float32).min, -1e31])
@pytest.mark.parametrize("cap", [0.0, 5.0])
@pytest.mark.parametrize("window,new,past,cut", [(50, [1, 200, 33, 65], [0, 0, 190, 63], False),
                                                 (1000, [300, 40], [1500, 900], True)])
def test_window_flash_heads_without_a_sink(window, new, past, cut, cap, sink):
    """A sink that weighs nothing beside ones that do, behind a window: a wave's later queries meet
    tiles of which they see no key, before and between the ones that they do see."""
    from enterprise_inference_amd.ops import attention as A
    from enterprise_inference_amd.ops import window_attention as wa
    H, G, D, bs, bf = 4, 1, 128, 64, torch.bfloat16
    g = torch.Generator().manual_seed(window)
    bt, n = _pages(g, [a + b for a, b in zip(new, past)], bs)
    cu = torch.tensor([0] + new).cumsum(0).to(torch.int32)
    pos = torch.cat([torch.arange(k) + f for k, f in zip(new, past)]).to(torch.int32)
    T = int(cu[-1])
    rnd = lambda *s: torch.randn(*s, generator=g).to(bf)
    q, k, v = rnd(T, H * D), rnd(n, bs, G * D), rnd(n, G * D, bs)

    def run(dev):
        md = A.AttentionMetadata(
            num_decode=0, num_prefill_tokens=T, slot_mapping=pos.to(dev), positions=pos.to(dev),
            prefill_block_tables=bt.to(dev), prefill_cu_q=cu.to(dev), prefill_q_lens=new)
        spec = wa.WindowSpec(H, G, 1, D, D, window, 0, mult=torch.full((H,), D ** -0.5).to(dev),
                             sink=torch.tensor([sink, 0.3, sink, -2.0]).to(dev), cap=cap)
        if dev == "cuda":
            qb = wa.query_block(spec, bf, bs)
            items = sum(-(-a // qb) for a in new)
            assert (wa.flash_parts(items, spec, qb, max(new), bt.shape[1] * bs)[0] > 1) == cut
        return wa.window_attention(q.to(dev), k.to(dev), v.to(dev), md, spec, None).cpu()

    a, b = run("cpu").double(), run("cuda").double()
    assert torch.isfinite(b).all()
    assert float((a - b).norm() / a.norm()) < 4e-3           # one bf16 rounding (2^-9) on each side


@pytest.mark.parametrize("kind", ["plain", "cap", "sigmoid", "pair"])
@pytest.mark.parametrize("D,Dv,bs", [(128, 128, 64), (72, 48, 32), (64, 112, 128)])
@pytest.mark.parametrize("parts", [1, 3])
def test_window_decode_slots_behind(parts, D, Dv, bs, kind, monkeypatch):
    """Cache slots behind a row's context hold anything: nothing of them reaches its output."""
    from enterprise_inference_amd.ops import attention as A
    from enterprise_inference_amd.ops import window_attention as wa
    monkeypatch.setenv("EIA_WINDOW_DECODE_P", str(parts))
    H, G, P, bf = 6, 2, 2 if kind == "pair" else 1, torch.bfloat16
    D = min(D, 64) if kind == "pair" else D
    g = torch.Generator().manual_seed(D + bs)
    lens = [1, 31, 33, 257, 700]
    bt, n = _pages(g, lens, bs)
    pos = torch.tensor(lens, dtype=torch.int32) - 1
    rnd = lambda *s: torch.randn(*s, generator=g).to(bf)
    q, k, v = rnd(len(lens), H * P * D), rnd(n, bs, G * P * D), rnd(n, G * Dv, bs)
    for s, m in enumerate(lens):
        last, used = int(bt[s, -(-m // bs) - 1]), (m - 1) % bs + 1
        k[last, used:], v[last, :, used:] = float("nan"), float("nan")

    def run(dev):
        md = A.AttentionMetadata(
            num_decode=len(lens), num_prefill_tokens=0, slot_mapping=pos.to(dev),
            positions=pos.to(dev), decode_block_tables=bt.to(dev), decode_seq_lens=(pos + 1).to(dev))
        return wa.window_attention(q.to(dev), k.to(dev), v.to(dev), md,
                                   _spec(wa, kind, H, G, D, Dv, 300, dev), None).cpu()

    a, b = run("cpu").double(), run("cuda").double()
    assert float((a - b).norm() / a.norm()) < 4e-3           # one bf16 rounding (2^-9) on each side


@pytest.mark.parametrize("H,G,D,Dv,bs", [(8, 2, 64, 128, 64), (3, 1, 40, 48, 64), (2, 2, 64, 80, 128)])
@pytest.mark.parametrize("window,keep,new,past", [(900, 5, [130, 1, 31], [1500, 0, 800]), (0, 0, [40, 700], [1000, 0])])
@pytest.mark.parametrize("parts", [0, 2, 7])                 # 0: the layer's own rule
def test_window_flash_pairs_in_parts(parts, window, keep, new, past, H, G, D, Dv, bs, monkeypatch):
    """Differential pairs whose keys are cut: both maps' parts, row blocks with fewer parts than others or one."""
    from enterprise_inference_amd.ops import attention as A
    from enterprise_inference_amd.ops import window_attention as wa
    if parts:
        monkeypatch.setattr(wa, "pair_parts", lambda n, sp, q, c: (parts, -(-(-(-c // 64)) // parts)))
    g, bf = torch.Generator().manual_seed(H + Dv), torch.bfloat16
    bt, n = _pages(g, [a + b for a, b in zip(new, past)], bs)
    cu = torch.tensor([0] + new).cumsum(0).to(torch.int32)
    pos = torch.cat([torch.arange(k) + f for k, f in zip(new, past)]).to(torch.int32)
    T = int(cu[-1])
    rnd = lambda *s: torch.randn(*s, generator=g).to(bf)
    q, k, v = rnd(T, H * 2 * D), rnd(n, bs, G * 2 * D), rnd(n, G * Dv, bs)

    def run(dev):
        md = A.AttentionMetadata(
            num_decode=0, num_prefill_tokens=T, slot_mapping=pos.to(dev), positions=pos.to(dev),
            prefill_block_tables=bt.to(dev), prefill_cu_q=cu.to(dev), prefill_q_lens=new)
        spec = wa.WindowSpec(H, G, 2, D, Dv, window, keep, mult=torch.full((2 * H,), D ** -0.5).to(dev))
        spec.epilogue, spec.eps, spec.post, spec.lam = 1, 1e-5, 0.7, torch.tensor([0.4]).to(dev)
        if dev == "cuda" and not parts:
            qb = wa.query_block(spec, bf, bs)
            assert wa.pair_parts(sum(-(-a // qb) for a in new), spec, qb, bt.shape[1] * bs)[0] > 1
        return wa.window_attention(q.to(dev), k.to(dev), v.to(dev), md, spec, None).cpu()

    a, b = run("cpu").double(), run("cuda").double()
    assert float((a - b).norm() / a.norm()) < 4e-3           # one bf16 rounding (2^-9) on each side
