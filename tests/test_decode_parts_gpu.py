"""Rows in key partitions, against the ops' own plain CPU path: rows that the grid is padded for, a padding
row, lengths where a row has one partition more or less, and more partitions than the merge takes at once."""

import pytest
import torch

from enterprise_inference_amd.ops import attention as A
from enterprise_inference_amd.ops import latent_attention as LA
from enterprise_inference_amd.ops import window_attention as WA

PAGE = 64


def _rel(a, b):
    a, b = a.double().cpu(), b.double().cpu()
    return float((a - b).norm() / b.norm())


def _step(lens, g):
    """Metadata of a decode step; a length of 0 is a padding row."""
    pages = [-(-max(n, 1) // PAGE) for n in lens]
    order = torch.randperm(sum(pages), generator=g).to(torch.int32)
    table = torch.zeros(len(lens), max(pages), dtype=torch.int32)
    at = 0
    for s, k in enumerate(pages):
        table[s, :k] = order[at:at + k]
        at += k
    i32 = lambda v: torch.tensor(v, dtype=torch.int32)
    return dict(slot_mapping=i32([0] * len(lens)), positions=i32([max(n - 1, 0) for n in lens]), num_seqs=len(lens),
                num_decode=len(lens), num_prefill_tokens=0, decode_block_tables=table, decode_seq_lens=i32(lens)), sum(pages)


def _both(call, tensors, md, lens):
    """On the CPU and on the GPU, live rows."""
    live = torch.tensor([n > 0 for n in lens])
    out = []
    for dev in ("cpu", "cuda"):
        m = A.AttentionMetadata(**{k: v.to(dev) if isinstance(v, torch.Tensor) else v for k, v in md.items()})
        out.append(call(dev, [None if t is None else t.to(dev) for t in tensors], m).cpu()[live])
    return out


LENS = {"edges": [1, 449, 480, 481, 512, 513, 544, 0, 2100, 3100], "one": [900], "few": [1500, 33, 1024]}


@pytest.mark.gpu
@pytest.mark.parametrize("parts", [0, 5, 23])
@pytest.mark.parametrize("lens", LENS.values(), ids=LENS.keys())
@pytest.mark.parametrize("kind,D,Dv,window", [("sink", 128, 128, 0), ("sigmoid", 96, 96, 500), ("pair", 64, 128, 1024),
                                              ("plain", 64, 64, 0)])
def test_window(kind, D, Dv, window, lens, parts, monkeypatch):
    monkeypatch.setenv("EIA_WINDOW_DECODE_P", str(parts))
    g = torch.Generator().manual_seed(len(lens) + D)
    H, G, P = 4, 2, 2 if kind == "pair" else 1
    md, pages = _step(lens, g)
    rnd = lambda *s: torch.randn(*s, generator=g)
    bf = lambda *s: rnd(*s).to(torch.bfloat16)
    q, k, v = bf(len(lens), H * P * D), bf(pages, PAGE, G * P * D), bf(pages, G * Dv, PAGE)
    sink, bias = rnd(H), torch.full((H,), -4.0)

    def call(dev, t, m):
        spec = WA.WindowSpec(H, G, P, D, Dv, window, 0, torch.full((H * P,), D ** -0.5, device=dev))
        if kind == "sink":
            spec.sink = t[3]
        elif kind == "sigmoid":
            spec.weights, spec.bias = 1, t[4]
        elif kind == "pair":
            spec.keep, spec.epilogue, spec.eps, spec.post, spec.lam = 4, 1, 1e-5, 0.7, torch.tensor([0.4], device=dev)
        return WA.window_attention(t[0], t[1], t[2], m, spec)

    # (a row of 3100 tokens: 24 partitions of four blocks, if there are so many)
    want, got = _both(call, [q, k, v, sink, bias], md, lens)
    # one rounding to bf16 on either side, 2^-9 / sqrt(3) each, and the products' order
    assert _rel(got, want) < 4e-3


@pytest.mark.gpu
@pytest.mark.parametrize("parts", [0, 5, 23])
@pytest.mark.parametrize("lens", [[1, 63, 64, 65, 128, 129, 0, 700, 2100], [900], [1500, 33, 1024]],
                         ids=["edges", "one", "few"])
@pytest.mark.parametrize("H,R,rd,window", [(8, 128, 32, 0), (20, 256, 32, 500), (16, 512, 64, 1024)])
def test_latent(H, R, rd, window, lens, parts, monkeypatch):
    monkeypatch.setenv("EIA_LATENT_DECODE_P", str(parts))
    g = torch.Generator().manual_seed(len(lens) + R)
    md, pages = _step(lens, g)
    bf = lambda *s: torch.randn(*s, generator=g).to(torch.bfloat16)
    t = [bf(len(lens), H, R), bf(len(lens), H, rd), bf(pages, PAGE, R + rd), bf(len(lens), H),
         torch.randn(H, generator=g) if window else None]

    def call(dev, t, m):
        return LA.latent_attention(t[0], t[1], LA.inv_frequencies(rd, 10000.0, dev), rd, t[2], m, t[3], (R + rd) ** -0.5,
                                   window, t[4])

    want, got = _both(call, t, md, lens)
    # as above, and the rotated queries' rounding to bf16 (2^-9 of a score of about one)
    assert _rel(got, want) < 8e-3


# heads on kv heads, rows: (row, kv head) pairs that do not fill eight XCDs, rows one XCD each does not hold
@pytest.mark.gpu
@pytest.mark.parametrize("H,G,rows", [(32, 8, 1), (8, 8, 3), (16, 4, 2), (6, 3, 9), (5, 5, 7), (12, 6, 20), (64, 32, 1), (8, 1, 1)])
def test_window_units(H, G, rows):
    g = torch.Generator().manual_seed(H + rows)
    lens = [1300 - 151 * (i % 8) for i in range(rows)]
    lens[rows // 2] = 0 if rows > 2 else 700
    md, pages = _step(lens, g)
    bf = lambda *s: torch.randn(*s, generator=g).to(torch.bfloat16)
    t = [bf(rows, H * 64), bf(pages, PAGE, G * 64), bf(pages, G * 64, PAGE), torch.randn(H, generator=g)]

    def call(dev, t, m):
        spec = WA.WindowSpec(H, G, 1, 64, 64, 0, 0, torch.full((H,), 0.125, device=dev))
        spec.sink = t[3]
        assert WA.decode_partitions(rows, spec) > 1
        return WA.window_attention(t[0], t[1], t[2], m, spec)

    want, got = _both(call, t, md, lens)
    assert _rel(got, want) < 4e-3                       # as in test_window


def test_window_partitions():
    """No more workgroups of an XCD's (row, kv head) pairs than its 32 CUs hold, none for what one workgroup does as fast,
    and no fewer than powers of two over the whole chip: few rows use every XCD."""
    spec = lambda w, G=2: WA.WindowSpec(4 * G, G, 1, 128, 128, w, 0, torch.ones(4 * G))
    assert [WA.decode_partitions(n, spec(1024)) for n in (1, 8, 9, 16, 17, 31, 64, 128)] == [8, 8, 8, 8, 6, 4, 2, 1]
    assert [WA.decode_partitions(n, spec(0)) for n in (1, 8, 9, 17, 128)] == [16, 16, 10, 6, 1]
    assert [WA.decode_partitions(3, spec(w)) for w in (300, 448, 449, 512)] == [1, 1, 4, 4]
    assert [WA.decode_partitions(n, spec(0, 8)) for n in (1, 2, 3, 4, 8)] == [16, 16, 10, 8, 4]
    for n in range(1, 300):
        for G in (1, 2, 3, 4, 6, 8, 16, 32):
            p, q = WA.decode_partitions(n, spec(0, G)), 1
            assert p == 1 or -(-n * G // 8) * p <= 32
            while 2 * q <= 16 and n * G * 2 * q <= 256:
                q *= 2
            assert p >= q


# rows whose partitions an XCD holds, whose last ones go beside the rows of others (1 to 7, 9, 13), or that are not padded
# (20 of four slices); and contexts that use more partitions than the merge takes at once
@pytest.mark.gpu
@pytest.mark.parametrize("H,R,rd,rows,ctx", [(16, 512, 64, 1, 4300), (8, 256, 64, 2, 4300), (16, 256, 64, 5, 3300),
                                             (64, 512, 64, 3, 1500), (8, 128, 32, 9, 4300), (20, 512, 64, 13, 900),
                                             (16, 320, 64, 13, 1400), (64, 320, 32, 20, 400), (128, 320, 0, 9, 300)])
def test_latent_places(H, R, rd, rows, ctx):
    g = torch.Generator().manual_seed(H + rows)
    lens = [max(1, ctx - 190 * (i % 8)) for i in range(rows)]
    if rows > 2:
        lens[rows // 2] = 0
    md, pages = _step(lens, g)
    bf = lambda *s: torch.randn(*s, generator=g).to(torch.bfloat16)
    t = [bf(rows, H, R), bf(rows, H, rd), bf(pages, PAGE, R + rd), bf(rows, H), torch.randn(H, generator=g)]

    def call(dev, t, m):
        return LA.latent_attention(t[0], t[1], LA.inv_frequencies(rd, 10000.0, dev), rd, t[2], m, t[3], (R + rd) ** -0.5,
                                   0, t[4])

    want, got = _both(call, t, md, lens)
    assert _rel(got, want) < 8e-3                       # as in test_latent


def test_latent_partitions():
    """At least nine tenths of the workgroups that the chip's CUs take at once (one each, two of narrow rows), never more."""
    assert [LA.decode_partitions(n, 16, window=1024) for n in (1, 8, 13, 24, 48, 100, 400)] == [17, 17, 17, 10, 5, 2, 1]
    assert [LA.decode_partitions(n, 8, wide=False) for n in (1, 13, 48, 100)] == [64, 39, 10, 5]
    assert [LA.decode_partitions(n, 64) for n in (1, 3, 9, 20, 65)] == [64, 21, 7, 3, 1]
    for n in range(1, 300):
        for H in (8, 16, 32, 64, 128):
            p, wgs = LA.decode_partitions(n, H), n * -(-H // 16)
            assert p == 1 or wgs * p <= 256
            assert p == 64 or 10 * p >= 9 * (256 // wgs)


@pytest.mark.gpu
@pytest.mark.parametrize("parts", [0, 2, 5, 16])                # 0: the layer's own rule
@pytest.mark.parametrize("H,G,D,window,keep", [(8, 2, 128, 100, 0), (16, 4, 64, 0, 0), (3, 1, 96, 300, 5), (6, 3, 32, 40, 0)])
@pytest.mark.parametrize("new,past", [([1, 40, 17], [0, 250, 31]), ([33], [300])], ids=["ragged", "one"])
def test_mixed_prefill(new, past, H, G, D, window, keep, parts, monkeypatch):
    if parts:
        monkeypatch.setattr(WA, "mix_parts", lambda *a: parts)
    g = torch.Generator().manual_seed(H + D)
    md, pages = _step([n + p for n, p in zip(new, past)], g)
    i32 = lambda v: torch.tensor(v, dtype=torch.int32)
    T, cu = sum(new), [0]
    for n in new:
        cu.append(cu[-1] + n)
    md = dict(md, num_decode=0, num_prefill_tokens=T, decode_block_tables=None, decode_seq_lens=None,
              positions=i32([p + i for n, p in zip(new, past) for i in range(n)]), prefill_cu_q=i32(cu),
              prefill_block_tables=md["decode_block_tables"], prefill_q_lens=new)
    rnd = lambda *s: torch.randn(*s, generator=g)
    bf = lambda *s: rnd(*s).to(torch.bfloat16)
    tensors = [bf(T, H * D), bf(pages, PAGE, G * D), bf(pages, G * D, PAGE), bf(T, H * D), rnd(H).abs() * 0.02,
               torch.eye(H) + 0.05 * rnd(H, H), rnd(H) if keep else None]

    def call(dev, t, m):
        spec = WA.WindowSpec(H, G, 1, D, D, window, keep, torch.full((H,), D ** -0.5, device=dev))
        spec.slope, spec.talk, spec.sink = t[4:]
        y = torch.full((T + 2, H * D), 7.0, dtype=torch.bfloat16, device=dev)      # two rows of no sequence
        rows = torch.cat([t[0], t[0][:2]])
        m.positions = torch.cat([m.positions, m.positions[:2]])
        WA.window_attention(rows, t[1], t[2], m, spec, torch.cat([t[3], t[3][:2]]), out=y)
        assert dev == "cpu" or bool((y[T:] == 7).all())
        return y[:T]

    ref, out = [], []
    for dev, to in (("cpu", ref), ("cuda", out)):
        m = A.AttentionMetadata(**{k: v.to(dev) if isinstance(v, torch.Tensor) else v for k, v in md.items()})
        to.append(call(dev, [None if t is None else t.to(dev) for t in tensors], m))
    assert torch.isfinite(out[0]).all() and _rel(out[0], ref[0]) < 2.0 ** -8 * 2      # two roundings to bf16
