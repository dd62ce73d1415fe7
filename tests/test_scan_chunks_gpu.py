"""Chunk-parallel recurrences against the ops' own plain CPU path, at the lengths where chunks and
their 8- and 16-token blocks begin and end."""

import pytest
import torch

pytestmark = pytest.mark.gpu

LENS = [[1, 64, 63, 65, 130], [200], [7, 9, 50, 47, 129, 1, 300]]


def _rel(a, b):
    a, b = a.double().cpu(), b.double().cpu()
    return float((a - b).norm() / b.norm())


def _step(lens, first, skip):
    """cu, positions (sequence s starts at first[s]) and slots (a skipped sequence: -1)."""
    cu = torch.tensor([0] + lens).cumsum(0).to(torch.int32)
    pos = torch.cat([torch.arange(n) + f for n, f in zip(lens, first)]).to(torch.int32)
    slots = torch.arange(len(lens)).flip(0).to(torch.int32)
    if skip:
        slots[1] = -1
    return cu, pos, slots


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("H,D", [(2, 64), (3, 40), (1, 16)])
@pytest.mark.parametrize("lens", LENS)
def test_wkv_chunks(lens, H, D, dtype):
    from enterprise_inference_amd.ops import wkv
    g = torch.Generator().manual_seed(sum(lens) + D)
    rnd = lambda *s: torch.randn(*s, generator=g)
    n, T, HD = len(lens), sum(lens), H * D
    assert max(lens) >= wkv.chunk_rows(n, H) and D <= wkv.CHUNK_DIM
    cu, pos, slots = _step(lens, [0 if s % 2 == 0 else 5 for s in range(n)], n > 3)
    r, k, v, gate = rnd(4, T, HD).mul(0.5).to(dtype)
    dec = rnd(T, HD)
    # decays from 0.998 a token down to channels that forget everything at once
    w0 = torch.linspace(-6.0, 4.0, HD).to(dtype)
    u, nw, x = rnd(HD).to(dtype), (1 + 0.1 * rnd(HD)).to(dtype), rnd(T, 24)
    S, prev = rnd(n, H, D, D), rnd(n, 24)
    args = [r, k, v, gate, dec, w0, u, nw, S, prev, x, slots, cu]
    dev = [t.to("cuda") for t in args]
    y = wkv.wkv_scan(*args, n, pos, None, 1e-5, H)
    z = wkv.wkv_scan(*dev, n, pos.to("cuda"), None, 1e-5, H)
    live = torch.cat([torch.full((m,), int(s) >= 0) for m, s in zip(lens, slots)])
    # fp32 sums over at most 64 products and a few exponentials; bf16 adds one rounding (2^-9)
    # and, where the two sides fall on different neighbours, one step more
    assert _rel(z.cpu()[live], y[live]) < (1e-5 if dtype == torch.float32 else 4e-3)
    assert _rel(dev[8], S) < 2e-6
    assert torch.equal(dev[9].cpu(), prev)
