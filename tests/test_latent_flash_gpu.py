"""The matrix-core forms of latent attention against the op's own plain CPU path: head counts that do
not fill a workgroup, every latent width class, pages smaller and larger than a key tile, windows,
contexts that are cut into parts."""

import pytest
import torch

pytestmark = pytest.mark.gpu


def _pages(g, total, bs):
    """Random pages for sequences of ``total`` tokens: block tables and the page count."""
    pages = [-(-n // bs) for n in total]
    order = torch.randperm(sum(pages), generator=g).to(torch.int32)
    bt = torch.zeros(len(total), max(pages), dtype=torch.int32)
    at = 0
    for s, n in enumerate(pages):
        bt[s, :n] = order[at:at + n]
        at += n
    return bt, sum(pages)


def _check(a, b):
    # both sides sum in fp32 and round once to bf16 (2^-9).  The kernels also round the rotated query
    # entries to bf16: rd of the R + rd products of a score (of order 1) off by 2^-9 each, weights
    # off by a few 1e-3, and an output by that part of the values' magnitude
    a, b = a.double(), b.double()
    assert float((a - b).norm() / a.norm()) < 4e-3
    assert float(((a - b).abs() / (a.abs() + a.abs().mean())).max()) < 2 ** -6


@pytest.mark.parametrize("H,R,rd", [(8, 128, 32), (3, 48, 16), (20, 40, 8), (16, 256, 32), (5, 200, 104),
                                    (8, 256, 72), (16, 512, 64), (2, 512, 128)])
@pytest.mark.parametrize("window,bs,new,past", [(0, 64, [1, 70, 33], [0, 0, 100]),
                                                (50, 128, [1, 70, 33], [0, 0, 100]),
                                                (0, 16, [65, 20], [0, 30]),
                                                (0, 64, [9], [1000])])
def test_latent_flash(window, bs, new, past, H, R, rd):
    from enterprise_inference_amd.ops import attention as A
    from enterprise_inference_amd.ops import latent_attention as la
    g = torch.Generator().manual_seed(H + R + window)
    bt, n = _pages(g, [a + b for a, b in zip(new, past)], bs)
    cu = torch.tensor([0] + new).cumsum(0).to(torch.int32)
    pos = torch.cat([torch.arange(k) + f for k, f in zip(new, past)]).to(torch.int32)
    T, bf = int(cu[-1]), torch.bfloat16
    rnd = lambda *s: torch.randn(*s, generator=g).to(bf)
    qa, qr, cache = rnd(T, H, R), rnd(T, H, rd), rnd(n, bs, R + rd)
    for s, k in enumerate([a + b for a, b in zip(new, past)]):   # slots behind a sequence hold anything
        cache[int(bt[s, -(-k // bs) - 1]), (k - 1) % bs + 1:] = float("nan")
    gate, sink = (rnd(T, H), None) if window == 0 else (None, torch.randn(H, generator=g))
    inv = la.inv_frequencies(rd, 100.0, "cpu")

    def run(dev):
        d = lambda t: None if t is None else t.to(dev)
        md = A.AttentionMetadata(
            num_decode=0, num_prefill_tokens=T, slot_mapping=d(pos), positions=d(pos),
            prefill_block_tables=d(bt), prefill_cu_q=d(cu), prefill_q_lens=new)
        return la.latent_attention(d(qa), d(qr), d(inv), rd - 8, d(cache), md, d(gate),
                                   (R + rd) ** -0.5, window, d(sink), bool(window), 1.1).cpu()

    _check(run("cpu"), run("cuda"))


@pytest.mark.parametrize("H,R,rd", [(8, 128, 32), (3, 48, 16), (20, 40, 8), (16, 256, 32), (8, 256, 64),
                                    (16, 512, 64), (2, 512, 128)])
@pytest.mark.parametrize("window,bs,parts", [(0, 64, 1), (0, 64, 3), (70, 128, 2), (0, 16, 64), (200, 48, 5)])
def test_latent_decode(window, bs, parts, H, R, rd, monkeypatch):
    from enterprise_inference_amd.ops import attention as A
    from enterprise_inference_amd.ops import latent_attention as la
    monkeypatch.setenv("EIA_LATENT_DECODE_P", str(parts))
    g = torch.Generator().manual_seed(H + R + window)
    total = [1, 64, 65, 300, 129]
    bt, n = _pages(g, total, bs)
    pos = torch.tensor(total, dtype=torch.int32) - 1
    T, bf = len(total), torch.bfloat16
    rnd = lambda *s: torch.randn(*s, generator=g).to(bf)
    qa, qr, cache = rnd(T, H, R), rnd(T, H, rd), rnd(n, bs, R + rd)
    for s, k in enumerate(total):
        cache[int(bt[s, -(-k // bs) - 1]), (k - 1) % bs + 1:] = float("nan")
    gate, sink = (rnd(T, H), None) if window == 0 else (None, torch.randn(H, generator=g))
    inv = la.inv_frequencies(rd, 100.0, "cpu")

    def run(dev):
        d = lambda t: None if t is None else t.to(dev)
        md = A.AttentionMetadata(
            num_decode=T, num_prefill_tokens=0, slot_mapping=d(pos), positions=d(pos),
            decode_block_tables=d(bt), decode_seq_lens=d(pos + 1))
        return la.latent_attention(d(qa), d(qr), d(inv), rd - 8, d(cache), md, d(gate),
                                   (R + rd) ** -0.5, window, d(sink), bool(window), 1.1).cpu()

    _check(run("cpu"), run("cuda"))
