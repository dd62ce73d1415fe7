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


@pytest.mark.parametrize("least", [1, 8, 10, 64])
@pytest.mark.parametrize("lens", [[9, 150, 8, 7, 63, 64, 65], [70, 9]])
def test_wkv_short_sequences_beside_a_long_one(lens, least, monkeypatch):
    """The same whichever of the two forms the shorter sequences take."""
    from enterprise_inference_amd.ops import wkv
    monkeypatch.setattr(wkv, "chunk_rows_beside", lambda n, h: least)
    n, T, H, D = len(lens), sum(lens), 2, 64
    cu, pos, slots = _step(lens, [3] * n, False)
    args = _wkv_args(torch.Generator().manual_seed(n), T, n, H, D, torch.float32) + [slots, cu]
    dev = [t.to("cuda") for t in args]
    y = wkv.wkv_scan(*args, n, pos, None, 1e-5, H)
    z = wkv.wkv_scan(*dev, n, pos.to("cuda"), None, 1e-5, H).cpu()
    # fp32 sums over at most 64 products and a few exponentials
    assert _rel(z, y) < 1e-5 and _rel(dev[8], args[8]) < 2e-6
    assert torch.equal(dev[9].cpu(), args[9])


# none of those that might be long is; one of many is; the average tells
@pytest.mark.parametrize("lens", [[20] * 12, [1] * 70 + [120] + [20] * 40, [28, 31, 52, 54, 19], [47, 100, 60], [30, 90]])
def test_wkv_lengths_not_told(lens):
    """The same where the longest sequence's rows are not given."""
    from enterprise_inference_amd.ops import wkv
    n, T, H, D = len(lens), sum(lens), 2, 64
    assert wkv.chunk_split(T, n, H) > 0
    cu, pos, slots = _step(lens, [3] * n, False)
    args = _wkv_args(torch.Generator().manual_seed(n), T, n, H, D, torch.float32) + [slots, cu]
    out = []
    for longest in (0, max(lens)):
        dev = [t.to("cuda") for t in args]
        out.append((wkv.wkv_scan(*dev, n, pos.to("cuda"), None, 1e-5, H, longest), dev[8], dev[9]))
    (y, S, prev), (y1, S1, prev1) = out
    # fp32 sums over at most 64 products and a few exponentials
    assert _rel(y, y1) < 1e-5 and _rel(S, S1) < 2e-6 and torch.equal(prev, prev1)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("mode,rot,half", [("exp_gates", 0, True), ("decay", 64, True),
                                           ("decay", 12, False), ("exp_gates", 20, True)])
@pytest.mark.parametrize("H,D,Dv", [(2, 128, 128), (3, 64, 64), (2, 72, 40)])
@pytest.mark.parametrize("lens", [[1, 128, 127, 129, 300], [500], [16, 15, 17, 144, 3]])
def test_linear_chunks(lens, H, D, Dv, mode, rot, half, dtype, monkeypatch):
    from enterprise_inference_amd.ops import linear_scan as ls
    monkeypatch.setattr(ls, "FORCE_CHUNKED", True)
    g = torch.Generator().manual_seed(sum(lens) + D + rot)
    rnd = lambda *s: torch.randn(*s, generator=g)
    n, T = len(lens), sum(lens)
    cu, pos, slots = _step(lens, [0 if s % 2 == 0 else 5 for s in range(n)], n > 3)
    at = [0, H * D, 2 * H * D, 2 * H * D + H * Dv, 2 * H * (D + Dv), 2 * H * (D + Dv) + H]
    x = rnd(T, at[-1] + H)
    x[:, at[-1]:] += 3.0
    x = x.to(dtype)
    inv = 10000.0 ** (-torch.arange(rot // 2) / max(1, rot // 2))

    def run(dev):
        spec = ls.ScanSpec(H, D, Dv, mode, cap=15.0, kscale=D ** -0.5, qscale=1.5, eps=1e-5,
                           rot_dims=rot, rot_half=half, inv_freq=inv.to(dev), out_scale=0.7,
                           decay=torch.linspace(0.999, 0.2, H).to(dev))
        st = ls.ScanState.allocate(n, spec, "cpu")
        gs = torch.Generator().manual_seed(1)
        for t in (st.S, st.n, st.m):
            if t is not None:
                t.copy_(torch.randn(t.shape, generator=gs))
        st = ls.ScanState(*(None if t is None else t.to(dev) for t in (st.S, st.n, st.m)))
        plan = ls.chunk_plan(lens, dev) if dev == "cuda" else None
        nw = torch.linspace(0.8, 1.2, H * Dv).to(dtype).to(dev)
        y = ls.linear_scan(x.to(dev), at[0], at[1], at[2], at[3], spec, st, slots.to(dev),
                           cu.to(dev), n, pos.to(dev), None, nw, at[4], at[5], plan=plan)
        return y.cpu(), st

    (y, a), (z, b) = run("cpu"), run("cuda")
    live = torch.cat([torch.full((m,), int(s) >= 0) for m, s in zip(lens, slots)])
    # fp32 sums over at most 128 products; bf16 adds one rounding and at times one step more
    assert _rel(z[live], y[live]) < (1e-5 if dtype == torch.float32 else 4e-3)
    for u, v in ((a.S, b.S), (a.n, b.n), (a.m, b.m)):
        assert u is None or _rel(v, u) < 2e-6


@pytest.mark.parametrize("lens", [[1024], [1025], [2048], [2049], [4100, 1]])
def test_gates_over_several_passes(lens, monkeypatch):
    """Edges of the passes in which the running maximum of the gates is formed.  The states forget within some
    hundred tokens (decays of about 0.95), so the bounds of short prompts hold."""
    test_linear_chunks(lens, 2, 16, 16, "exp_gates", 0, True, torch.float32, monkeypatch)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("lens", [[300, 128, 63, 65], [64, 129, 1, 400]])
def test_gates_that_shut(lens, dtype, monkeypatch):
    """Tokens, and whole chunks, that add nothing (an input gate of -inf), before and behind others, and tokens that
    forget almost everything: the maximum of a chunk's own gates is then none, or lies far below the one carried in."""
    from enterprise_inference_amd.ops import linear_scan as ls
    monkeypatch.setattr(ls, "FORCE_CHUNKED", True)
    H, D, Dv, n, T = 3, 32, 64, len(lens), sum(lens)
    g = torch.Generator().manual_seed(T)
    cu, pos, slots = _step(lens, [0, 5, 0, 7], False)
    at = [0, H * D, 2 * H * D, 2 * H * D + H * Dv, 2 * H * (D + Dv), 2 * H * (D + Dv) + H]
    x = torch.randn(T, at[-1] + H, generator=g)
    x[:, at[5]:] += 3.0
    x[::7, at[5]] = -30.0                                  # forgets
    x[3::5, at[4] + 1] = float("-inf")                     # adds nothing
    for lo in cu[:-1].tolist():
        x[lo:lo + 2, at[4]:at[5]] = float("-inf")          # nor do the first two
    x[cu[0] + 128:cu[0] + 256, at[4] + 2] = float("-inf")  # nor does a chunk of the first sequence, head 2
    x = x.to(dtype)
    (y, a), (z, b) = (_gated(dev, x, lens, cu, pos, slots, H, D, Dv) for dev in ("cpu", "cuda"))
    assert torch.isfinite(y).all() and _rel(z, y) < (1e-5 if dtype == torch.float32 else 4e-3)      # as above
    for u, v in ((a.S, b.S), (a.n, b.n), (a.m, b.m)):
        assert _rel(v, u) < 2e-6


def _gated(dev, x, lens, cu, pos, slots, H, D, Dv):
    """Matrix memory without a cap over rows of queries, keys, values, output gates and the two gates of each head."""
    from enterprise_inference_amd.ops import linear_scan as ls
    spec = ls.ScanSpec(H, D, Dv, "exp_gates", kscale=D ** -0.5, eps=1e-5)
    st = ls.ScanState.allocate(len(lens), spec, "cpu")
    gs = torch.Generator().manual_seed(1)
    for t in (st.S, st.n, st.m):
        t.copy_(torch.randn(t.shape, generator=gs))
    st = ls.ScanState(*(t.to(dev) for t in (st.S, st.n, st.m)))
    plan = ls.chunk_plan(lens, dev) if dev == "cuda" else None
    HD = H * D
    y = ls.linear_scan(x.to(dev), 0, HD, 2 * HD, 2 * HD + H * Dv, spec, st, slots.to(dev), cu.to(dev), len(lens),
                       pos.to(dev), None, None, 2 * H * (D + Dv), 2 * H * (D + Dv) + H, plan=plan)
    return y.cpu(), st


# first and last rows of a chunk, of the half that a wave takes, of a block of sixteen, of the sequence
@pytest.mark.parametrize("row", [0, 1, 63, 64, 127, 128, 130, 299])
@pytest.mark.parametrize("past", [0, 5])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("i,f,lead", [(float("-inf"), float("-inf"), 0), (float("-inf"), float("-inf"), 2),
                                      (0.5, float("-inf"), 0), (float("nan"), 1.0, 0), (float("nan"), 1.0, 2),
                                      (0.5, float("nan"), 0), (float("-inf"), float("nan"), 0), (float("inf"), 1.0, 0)])
def test_gates_that_are_not_finite(i, f, lead, dtype, past, row, monkeypatch):
    """One token's gates of head 1, behind ``lead`` tokens that add nothing.  A token that forgets everything and adds
    nothing, and one with a gate that is no number, leave none, as in the recurrence, in their own and all later outputs and in
    the state."""
    from enterprise_inference_amd.ops import linear_scan as ls
    monkeypatch.setattr(ls, "FORCE_CHUNKED", True)
    H, D, Dv, lens = 3, 32, 64, [300, 150]
    cu, pos, slots = _step(lens, [past, 5], False)
    at = 2 * H * (D + Dv)
    x = torch.randn(sum(lens), at + 2 * H, generator=torch.Generator().manual_seed(row))
    x[:, at + H:] += 3.0
    x[max(0, row - lead):row, at + 1] = float("-inf")
    x[row, at + 1], x[row, at + H + 1] = i, f
    x = x.to(dtype)
    (y, a), (z, b) = (_gated(dev, x, lens, cu, pos, slots, H, D, Dv) for dev in ("cpu", "cuda"))
    bad = torch.zeros(sum(lens), H, Dv, dtype=torch.bool)
    same = ~bad
    if not (i == 0.5 and f == float("-inf")):
        bad[row:lens[0], 1] = True
        same[row // 16 * 16:lens[0], 1] = False            # (a block of sixteen is one product)
    bad, same = bad.view(y.shape), same.view(y.shape)
    assert torch.equal(torch.isfinite(y), ~bad) and not torch.isfinite(z[bad]).any()
    assert torch.isfinite(z[same]).all() and _rel(z[same], y[same]) < (1e-5 if dtype == torch.float32 else 4e-3)  # as above
    for u, v in ((a.S, b.S), (a.n, b.n), (a.m, b.m)):
        v, ok = v.cpu(), torch.isfinite(u)
        assert u is a.m and (i != i or f != f) or torch.equal(torch.isfinite(v), ok)      # (maxima pass over NaN)
        assert _rel(v[ok], u[ok]) < 2e-6


def _stays_not_finite(y, z, H, col, hit):
    """What the recurrence (y) leaves not finite does not come out as a number (z), and where both are numbers they are
    the same.  col: an infinite value is one number of its column, (q . k) v, in sums over tokens, and a sum of infinities of
    both signs, none, in ones over the state's rows; the other columns are divided by its norm, to 0 or to no
    number.  So only that column is compared."""
    rows = lambda t: t.double().view(t.shape[0], H, -1)
    a, b = rows(y), rows(z)
    bad = ~torch.isfinite(a)
    assert bool(bad.any()) == hit
    if col is not None:
        a, b, bad = a[:, :, col], b[:, :, col], bad[:, :, col]
        assert bad.any()
    assert not torch.isfinite(b[bad]).any()
    ok = ~bad & torch.isfinite(b)
    assert ok.any() and _rel(b[ok], a[ok]) < 4e-3


@pytest.mark.parametrize("mode,rot", [("exp_gates", 0), ("decay", 64)])
@pytest.mark.parametrize("H,D,Dv", [(2, 128, 128), (2, 64, 64), (2, 72, 40)])
@pytest.mark.parametrize("where,value", [("v", float("inf")), ("v", float("nan")), ("k", float("-inf")),
                                         ("q", float("inf")), ("S", float("inf")), ("", 0.0)])
def test_linear_rows_that_are_not_finite(where, value, H, D, Dv, mode, rot, monkeypatch):
    """One entry of head 1 that is not finite stays where the recurrence leaves it."""
    from enterprise_inference_amd.ops import linear_scan as ls
    monkeypatch.setattr(ls, "FORCE_CHUNKED", True)
    g = torch.Generator().manual_seed(D + rot)
    lens, hit = [200, 150], 70                 # row 70 of the first sequence
    T = sum(lens)
    cu, pos, slots = _step(lens, [5, 0], False)
    at = [0, H * D, 2 * H * D, 2 * H * D + H * Dv, 2 * H * (D + Dv), 2 * H * (D + Dv) + H]
    x = torch.randn(T, at[-1] + H, generator=g)
    x[:, at[-1]:] += 3.0
    S0 = torch.randn(2, H, D, Dv, generator=g)
    if where == "S":
        S0[slots[0], 1, 3, 5] = value
    elif where:
        x[hit, at["qkv".index(where)] + (Dv if where == "v" else D) + 5] = value
    x = x.to(torch.bfloat16)
    inv = 10000.0 ** (-torch.arange(rot // 2) / max(1, rot // 2))

    def run(dev):
        spec = ls.ScanSpec(H, D, Dv, mode, cap=15.0, kscale=D ** -0.5, eps=1e-5, rot_dims=rot, rot_half=True,
                           inv_freq=inv.to(dev), decay=torch.linspace(0.999, 0.9, H).to(dev))
        st = ls.ScanState.allocate(2, spec, dev)
        st.S.copy_(S0)
        plan = ls.chunk_plan(lens, dev) if dev == "cuda" else None
        y = ls.linear_scan(x.to(dev), at[0], at[1], at[2], at[3], spec, st, slots.to(dev), cu.to(dev), 2,
                           pos.to(dev), None, None, at[4], at[5], plan=plan)
        return y.cpu().double(), st.S.cpu().double()

    (y, S), (z, R) = run("cpu"), run("cuda")
    live = torch.isfinite(S)
    assert bool(live.all()) == (where in ("", "q"))
    assert torch.equal(torch.isfinite(R), live)
    assert _rel(R[live], S[live]) < 2e-6
    # outputs of the other head, of the other sequence, and before the row's block of sixteen; a query is its row's own
    same = torch.ones(T, H, Dv, dtype=torch.bool)
    if where == "q":
        same[hit, 1] = False
    elif where:
        same[0 if where == "S" else hit // 16 * 16:lens[0], 1] = False
    same = same.view(T, H * Dv)
    assert torch.isfinite(z[same]).all() and _rel(z[same], y[same]) < 4e-3
    _stays_not_finite(y, z, H, 5 if value == float("inf") and where == "v" else None, where != "")


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("H,G,D,Dv", [(4, 2, 128, 128), (2, 2, 64, 64), (3, 1, 72, 40),
                                      (2, 1, 16, 120), (2, 2, 112, 6)])
@pytest.mark.parametrize("lens", [[1, 64, 63, 65, 130], [200], [15, 16, 17, 129, 3]])
def test_delta_chunks(lens, H, G, D, Dv, dtype, monkeypatch):
    y, S, z, Z, live = _delta_chunks(lens, H, G, D, Dv, dtype, monkeypatch)
    # fp32 sums over at most 128 products and a 64-row triangular solve; bf16 adds one rounding and
    # at times one step more
    assert _rel(z[live], y[live]) < (1e-5 if dtype == torch.float32 else 4e-3)
    assert _rel(Z, S) < 4e-6


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("lens,H,G,D,Dv", [([1, 64, 63, 65, 130], 16, 4, 128, 128), ([70] * 9, 8, 8, 64, 120),
                                           ([129, 150, 1, 16], 18, 2, 40, 64), ([65] * 8, 9, 9, 128, 33)])
def test_delta_chunks_many_heads(lens, H, G, D, Dv, dtype, monkeypatch):
    """More columns than CUs: 32 a workgroup; and more than eight heads to a key head."""
    y, S, z, Z, live = _delta_chunks(lens, H, G, D, Dv, dtype, monkeypatch)
    assert _rel(z[live], y[live]) < (1e-5 if dtype == torch.float32 else 4e-3)      # as above
    assert _rel(Z, S) < 4e-6


@pytest.mark.parametrize("lens,H,G,D,Dv", [([129, 64], 8, 1, 128, 128), ([129, 64], 10, 2, 64, 64), ([100], 48, 3, 16, 16),
                                           ([1] * 520, 9, 1, 16, 16), ([1] * 150 + [70] * 25, 18, 1, 16, 32),
                                           ([66] * 45, 20, 4, 40, 24)])
def test_delta_chunks_few_key_heads(lens, H, G, D, Dv, monkeypatch):
    """A key head's heads one to a workgroup, in parts (of two and more than eight heads), or all in one."""
    y, S, z, Z, live = _delta_chunks(lens, H, G, D, Dv, torch.float32, monkeypatch)
    assert _rel(z[live], y[live]) < 1e-5 and _rel(Z, S) < 4e-6                      # as above


@pytest.mark.parametrize("H,G,D,Dv", [(4, 2, 128, 128), (8, 4, 64, 72), (32, 8, 128, 128)])
@pytest.mark.parametrize("e,most", [(60, 0.0), (100, 2.0 ** -25), (-110, 2.0 ** -25)])
def test_delta_of_small_and_large_magnitudes(e, most, H, G, D, Dv, monkeypatch):
    """Values and state times 2^-e: so is the state after them.  At 2^-100 what falls below the smallest normal
    number is 2^-26 of the rest; times 2^110 overflows the parts, which fp32 products take over."""
    def run(scale):
        def plant(rows, S):
            rows[2].mul_(scale)
            S.mul_(scale)
        return _delta_chunks([150, 200], H, G, D, Dv, torch.float32, monkeypatch, plant)[3].double() / scale

    S, Z = run(1.0), run(2.0 ** -e)
    assert float((Z - S).norm() / S.norm()) <= (most if e > 0 else 4e-6)            # (other products: as above)


def test_delta_chunks_allocate_once(monkeypatch):
    """The workspaces of a step are one allocation beside its outputs: more of them show in short prompts."""
    from enterprise_inference_amd.ops import delta_scan as ds
    seen, empty = [], torch.empty

    def counted(*a, **k):
        seen.extend([a] if str(k.get("device")).startswith("cuda") else [])
        return empty(*a, **k)

    monkeypatch.setattr(ds.torch, "empty", counted)
    _, _, z, _, _ = _delta_chunks([100], 4, 2, 64, 64, torch.bfloat16, monkeypatch)
    assert torch.isfinite(z).all() and len(seen) == 2 + 1          # (one in the helper)


def _delta_chunks(lens, H, G, D, Dv, dtype, monkeypatch, plant=lambda rows, S: None):
    from types import SimpleNamespace
    from enterprise_inference_amd.ops import delta_scan as ds
    monkeypatch.setattr(ds, "FORCE_CHUNKED", True)
    g = torch.Generator().manual_seed(sum(lens) + D)
    rnd = lambda *s: torch.randn(*s, generator=g)
    n, T = len(lens), sum(lens)
    cu, pos, slots = _step(lens, [0 if s % 2 == 0 else 5 for s in range(n)], n > 3)
    pad = lambda t, m: torch.nn.functional.pad(t, (0, -(-m // 16) * 16 - m))
    unit = lambda t: t / t.norm(dim=-1, keepdim=True)
    rows = [pad(unit(rnd(T, G, D)), D), pad(unit(rnd(T, G, D)), D), pad(rnd(T, H, Dv), Dv),
            -torch.rand(T, H, generator=g) ** 4, torch.sigmoid(2.0 * rnd(T, H)),
            rnd(T, H * Dv).to(dtype)]
    S0, nw = rnd(n, H, D, Dv), (1 + 0.1 * rnd(Dv)).to(dtype)
    plant(rows, S0)

    def run(dev):
        md = SimpleNamespace(seq_cu=cu.to(dev), seq_slots=slots.to(dev), positions=pos.to(dev),
                             num_seqs=n, num_decode=0, num_prefill_tokens=T, prefill_q_lens=lens,
                             decode_seq_lens=None, work_cache={})
        st = ds.DeltaState(S0.clone().to(dev), None)
        spec = ds.DeltaSpec(H, G, D, Dv, 1, eps=1e-6, out_scale=0.7)
        plan = ds.prefill_plan(md, torch.device(dev)) if dev == "cuda" else None
        wide = torch.empty(T, H * Dv + 1, dtype=dtype, device=dev)      # rows of any alignment
        y = ds.delta_scan(ds.DeltaRows(*(t.to(dev) for t in rows)), spec, st, md, nw.to(dev),
                          wide[:, 1:] if D == 128 and n == 1 else None, plan)
        return y.cpu(), st.S.cpu()

    (y, S), (z, Z) = run("cpu"), run("cuda")
    live = torch.cat([torch.full((m,), int(s) >= 0) for m, s in zip(lens, slots)])
    return y, S, z, Z, live


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_delta_gates_that_are_nearly_shut(dtype, monkeypatch):
    """silu(-88) is -5e-37: the output is small, and not zero, though 1 / (1 + exp(88)) is below the smallest normal number."""
    cols = [0, 1, 70, 200]

    def plant(rows, S):
        rows[5][:, cols] = torch.tensor([-88.5, -88.0, -87.5, -60.0]).to(dtype)

    y, _, z, _, live = _delta_chunks([100, 64, 3], 2, 1, 128, 128, dtype, monkeypatch, plant)
    for c in cols:                                         # the bounds of test_delta_chunks
        u, v = y[live][:, c], z[live][:, c]
        ok = u.abs() > 2.0 ** -125                         # (the kernels flush numbers below 2^-126 to zero)
        assert ok.sum() > 100 and _rel(v[ok], u[ok]) < (1e-5 if dtype == torch.float32 else 4e-3)


@pytest.mark.parametrize("H,G,D,Dv", [(4, 2, 128, 128), (3, 3, 64, 72), (32, 8, 128, 128)])
@pytest.mark.parametrize("where,value", [("v", float("inf")), ("v", float("nan")), ("k", float("nan")),
                                         ("q", float("inf")), ("q", float("nan")), ("S", float("-inf")),
                                         ("v", 3.4e38), ("", 0.0)])
def test_delta_rows_that_are_not_finite(where, value, H, G, D, Dv, monkeypatch):
    """One entry of the last (key) head that is not finite stays where the recurrence leaves it."""
    lens, hit = [150, 200], 70                 # row 70 of the second sequence, past that which is its state's

    def plant(rows, S):
        if where == "S":
            S[0, H - 1, 3, 5] = value          # (slots run backwards)
        elif where:
            rows["qkv".index(where)][lens[0] + hit, -1, 5] = value

    y, S, z, Z, _ = _delta_chunks(lens, H, G, D, Dv, torch.bfloat16, monkeypatch, plant)
    fine, ok = torch.isfinite(S), torch.isfinite(y) & torch.isfinite(z)
    if value != 3.4e38:                        # (at the edge of fp32's range the order of sums decides)
        _stays_not_finite(y, z, H, 5 if value == float("inf") and where == "v" else None, where != "")
    assert torch.equal(torch.isfinite(Z), fine)
    assert _rel(z[ok], y[ok]) < 4e-3 and _rel(Z[fine], S[fine]) < 4e-6              # as above
    first = H - (1 if where in ("v", "S") else H // G)                  # heads that meet it
    same = torch.ones(sum(lens), H, Dv, dtype=torch.bool)
    if where:                                                           # (products take 16 tokens at a time)
        lo = lens[0] + (0 if where == "S" else hit if where == "q" else hit // 16 * 16)
        same[lo:lo + 1 if where == "q" else None, first:] = False
    assert torch.isfinite(z)[same.view(sum(lens), H * Dv)].all()


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("H,D,Dv,R,rot", [(2, 64, 128, 16, 0), (3, 32, 64, 33, 0), (2, 64, 64, 8, 64),
                                          (2, 24, 40, 5, 8), (1, 20, 126, 16, 6)])
@pytest.mark.parametrize("lens", [[1, 64, 63, 65, 130], [200], [7, 8, 9, 50, 129, 3]])
def test_channel_chunks(lens, H, D, Dv, R, rot, dtype, monkeypatch):
    from enterprise_inference_amd.ops import linear_scan as ls
    monkeypatch.setattr(ls, "FORCE_CHUNKED", True)
    g = torch.Generator().manual_seed(sum(lens) + D + R)
    rnd = lambda *s: torch.randn(*s, generator=g)
    n, T = len(lens), sum(lens)
    cu, pos, slots = _step(lens, [0 if s % 2 == 0 else 5 for s in range(n)], n > 3)
    at = [0, H * D, 2 * H * D, 2 * H * D + H * Dv, 2 * H * (D + Dv)]
    x = rnd(T, at[-1] + R).to(dtype)
    a2t, a2b = rnd(R, H * D), torch.linspace(-8.0, 8.0, H * D)     # from forgetting to keeping
    inv = 10000.0 ** (-torch.arange(rot // 2) / max(1, rot // 2))
    S0, nw = rnd(n, H, D, Dv), (1 + 0.1 * rnd(Dv)).to(dtype)

    def run(dev):
        spec = ls.ScanSpec(H, D, Dv, "channel", kscale=0.5, qscale=1.5, eps=1e-5, rot_dims=rot,
                           rot_half=rot != 8, inv_freq=inv.to(dev), out_scale=0.7, norm_shared=True,
                           a2t=a2t.to(dev), a2b=a2b.to(dev), tau=2.0)
        st = ls.ScanState.allocate(n, spec, "cpu")
        st = ls.ScanState(S0.clone().to(dev), None, None)
        plan = ls.chunk_plan(lens, dev) if dev == "cuda" else None
        y = ls.linear_scan(x.to(dev), at[0], at[1], at[2], at[3], spec, st, slots.to(dev),
                           cu.to(dev), n, pos.to(dev), None, nw.to(dev), lo_off=at[4], plan=plan)
        return y.cpu(), st.S.cpu()

    (y, S), (z, Z) = run("cpu"), run("cuda")
    live = torch.cat([torch.full((m,), int(s) >= 0) for m, s in zip(lens, slots)])
    # fp32 sums over at most 64 products, logarithms of decays summed over at most 64 tokens; bf16
    # adds one rounding and at times one step more
    assert _rel(z[live], y[live]) < (2e-5 if dtype == torch.float32 else 4e-3)
    assert _rel(Z, S) < 4e-6


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("mode", ["decay", "exp_gates", "channel"])
@pytest.mark.parametrize("H,D,Dv,rot", [(2, 64, 64, 0), (3, 64, 128, 64), (2, 128, 128, 0),
                                        (1, 72, 40, 12), (2, 17, 100, 0), (2, 64, 6, 0)])
def test_linear_decode_rows(H, D, Dv, rot, mode, dtype):
    from enterprise_inference_amd.ops import linear_scan as ls
    g = torch.Generator().manual_seed(D + Dv)
    rnd = lambda *s: torch.randn(*s, generator=g)
    n, R = 5, 9
    pos = torch.tensor([0, 7, 300, 4, 0], dtype=torch.int32)
    slots = torch.tensor([3, 0, -1, 4, 1], dtype=torch.int32)
    lens = torch.tensor([1, 8, 301, 0, 1], dtype=torch.int32)      # (0: a padding row)
    at = [0, H * D, 2 * H * D, 2 * H * D + H * Dv, 2 * H * (D + Dv), 2 * H * (D + Dv) + H]
    x = rnd(n, at[-1] + H + R).to(dtype)
    inv = 10000.0 ** (-torch.arange(rot // 2) / max(1, rot // 2))
    S0, N0, M0, nw = rnd(n, H, D, Dv), rnd(n, H, D), rnd(n, H), (1 + 0.1 * rnd(H * Dv)).to(dtype)
    a2t, a2b = rnd(R, H * D), rnd(H * D)

    def run(dev):
        spec = ls.ScanSpec(H, D, Dv, mode, cap=15.0, kscale=D ** -0.5, qscale=1.5, eps=1e-5,
                           rot_dims=rot, rot_half=rot != 12, inv_freq=inv.to(dev), out_scale=0.7,
                           decay=torch.linspace(0.999, 0.2, H).to(dev), a2t=a2t.to(dev),
                           a2b=a2b.to(dev), tau=2.0)
        st = ls.ScanState(*(t.clone().to(dev) if i == 0 or mode == "exp_gates" else None
                            for i, t in enumerate((S0, N0, M0))))
        y = ls.linear_scan(x.to(dev), at[0], at[1], at[2], at[3], spec, st, slots.to(dev), None, n,
                           pos.to(dev), lens.to(dev), nw.to(dev), at[4], at[5], lo_off=at[5] + H)
        return y.cpu(), st

    (y, a), (z, b) = run("cpu"), run("cuda")
    live = (slots >= 0) & (lens > 0)
    # fp32 sums over at most 128 products; bf16 adds one rounding and at times one step more
    assert _rel(z[live], y[live]) < (1e-5 if dtype == torch.float32 else 4e-3)
    for u, v in ((a.S, b.S), (a.n, b.n), (a.m, b.m)):
        if u is not None:                  # (a padding row leaves its slot alone on the GPU)
            kept = slots[live].long()
            assert _rel(v.cpu()[kept], u[kept]) < 2e-6
            if dtype == torch.float32 and u is a.S:
                assert torch.equal(v.cpu()[4], S0[4])


def _wkv_args(g, T, n, H, D, dtype):
    """Everything that wkv_scan takes before ``slots``; decays from 0.998 a token to about 0.4."""
    rnd = lambda *s: torch.randn(*s, generator=g)
    HD = H * D
    r, k, v, gate = rnd(4, T, HD).mul(0.5).to(dtype)
    w0, u, nw = torch.linspace(-6.0, -0.1, HD), rnd(HD), 1 + 0.1 * rnd(HD)
    return [r, k, v, gate, 0.3 * rnd(T, HD), w0.to(dtype), u.to(dtype), nw.to(dtype),
            rnd(n, H, D, D), rnd(n, 24), rnd(T, 24)]


@pytest.mark.parametrize("cu", [[0, 40], [20, 60], [0, 0], [70, 71], [3, 99], [50, 100]])
def test_wkv_sequence_of_a_wider_step(cu):
    """One sequence that owns some of the step's rows, on both sides of the length from which
    sequences are cut into chunks."""
    from enterprise_inference_amd.ops import wkv
    H, D, T = 2, 64, 100
    assert T >= wkv.chunk_rows(1, H) > 40
    args = _wkv_args(torch.Generator().manual_seed(cu[1]), T, 1, H, D, torch.float32)
    args += [torch.zeros(1, dtype=torch.int32), torch.tensor(cu, dtype=torch.int32)]
    pos = (torch.arange(T) + 5 - cu[0]).to(torch.int32)
    dev = [t.to("cuda") for t in args]
    y = wkv.wkv_scan(*args, 1, pos, None, 1e-5, H)
    z = wkv.wkv_scan(*dev, 1, pos.to("cuda"), None, 1e-5, H).cpu()
    # fp32 sums over at most 64 products and a few exponentials
    rows = slice(*cu)
    assert cu[0] == cu[1] or _rel(z[rows], y[rows]) < 1e-5
    assert _rel(dev[8], args[8]) < 2e-6
    assert torch.equal(dev[9].cpu(), args[9])


@pytest.mark.parametrize("value", [float("inf"), float("nan")])
@pytest.mark.parametrize("at", [0, 5, 15, 16, 70, 127, 129])
def test_wkv_values_that_are_not_finite(at, value):
    """A value that is no number reaches its own token and later ones, in its own head, only."""
    from enterprise_inference_amd.ops import wkv
    H, D, T = 2, 64, 130
    args = _wkv_args(torch.Generator().manual_seed(at), T, 1, H, D, torch.float32)
    clean = [t.to("cuda") for t in args]
    args[2][at, D + 7] = value
    bad = [t.to("cuda") for t in args]
    rest = [torch.zeros(1, dtype=torch.int32).cuda(), torch.tensor([0, T], dtype=torch.int32).cuda()]
    pos = torch.arange(T, dtype=torch.int32).cuda()
    y = wkv.wkv_scan(*clean, *rest, 1, pos, None, 1e-5, H)
    z = wkv.wkv_scan(*bad, *rest, 1, pos, None, 1e-5, H)
    # (the chunk's own sums are taken in another order: 16 fp32 products)
    assert torch.equal(y[:, :D], z[:, :D]) and (at == 0 or _rel(z[:at], y[:at]) < 1e-6)
    assert not torch.isfinite(z[at, D + 7]) and torch.isfinite(y).all()
    S, Z = clean[8][0], bad[8][0]                        # the head's column 7, and nothing else
    assert not torch.isfinite(Z[1, :, 7]).any()
    Z[1, :, 7] = S[1, :, 7]
    assert torch.equal(S, Z)


@pytest.mark.parametrize("every", [2, 3, 5])
def test_wkv_strongly_forgetting_tokens(every):
    """Channels that some tokens forget almost at once (2^-30 and less) and others keep: weights of
    the pairs behind such a token stay as exact as fp32 products of the decays."""
    from enterprise_inference_amd.ops import wkv
    H, D, T = 2, 64, 128
    g = torch.Generator().manual_seed(every)
    args = _wkv_args(g, T, 1, H, D, torch.float32)
    args[5] = torch.zeros(H * D)
    dec = torch.full((T, H * D), -6.0) + torch.rand(T, H * D, generator=g)
    dec[torch.rand(T, H * D, generator=g) < 1 / every] = 3.4
    args[4] = dec
    pos = torch.arange(T, dtype=torch.int32)
    dev = [t.to("cuda") for t in args]
    z = wkv.wkv_scan(*dev, torch.zeros(1, dtype=torch.int32).cuda(),
                     torch.tensor([0, T], dtype=torch.int32).cuda(), 1, pos.cuda(), None, 1e-5, H)
    r, k, v, gate = (t.double().view(T, H, D) for t in args[:4])
    w = torch.exp(-torch.exp(dec.double())).view(T, H, D)
    u, nw, S = args[6].double().view(H, D), args[7].double(), torch.zeros(H, D, D, dtype=torch.float64)
    y = torch.empty(T, H, D, dtype=torch.float64)
    for t in range(T):
        kv = k[t][:, :, None] * v[t][:, None]
        o = ((S + u[:, :, None] * kv) * r[t][:, :, None]).sum(1)
        S = w[t][:, :, None] * S + kv
        y[t] = o / torch.sqrt((o * o).mean(-1, keepdim=True) + 1e-5)
    y = y.flatten(1) * nw * torch.nn.functional.silu(gate.flatten(1))
    # 2^-23 and less each for the exponent, exp and product of a weight and for the sums: token by token
    # outputs are 1.4e-7 off; exponents that differ by an ulp of 160, the sum of four such decays, 8e-7
    assert _rel(z, y) < 3e-7
    assert _rel(dev[8][0], S) < 3e-7


@pytest.mark.parametrize("spread", [3.0, 8.0, 20.0])
def test_channel_strongly_forgetting_tokens(spread, monkeypatch):
    """As above for a decay per key channel, which a token's own entry passes too."""
    from enterprise_inference_amd.ops import linear_scan as ls
    H, D, Dv, R, T = 2, 64, 64, 16, 128
    g = torch.Generator().manual_seed(int(spread))
    rnd = lambda *s: torch.randn(*s, generator=g)
    at = [0, H * D, 2 * H * D, 2 * H * D + H * Dv, 2 * H * (D + Dv)]
    x, a2t, a2b = rnd(T, at[-1] + R), spread * rnd(R, H * D), torch.full((H * D,), 6.0)
    spec = ls.ScanSpec(H, D, Dv, "channel", kscale=D ** -0.5, eps=1e-5, a2t=a2t.cuda(), a2b=a2b.cuda(), tau=1.0)
    st = ls.ScanState(torch.zeros(1, H, D, Dv, device="cuda"), None, None)
    i32 = lambda v: torch.tensor(v, dtype=torch.int32, device="cuda")
    monkeypatch.setattr(ls, "FORCE_CHUNKED", True)
    y = ls.linear_scan(x.cuda(), at[0], at[1], at[2], at[3], spec, st, i32([0]), i32([0, T]), 1,
                       torch.arange(T, dtype=torch.int32).cuda(), plan=ls.chunk_plan([T], "cuda"),
                       lo_off=at[4])
    f = x.double()
    q, k = f[:, :H * D].view(T, H, D), f[:, H * D:2 * H * D].view(T, H, D) * D ** -0.5
    v, gate = f[:, at[2]:at[3]].view(T, H, Dv), f[:, at[3]:at[4]]
    a = torch.sigmoid(f[:, at[4]:] @ a2t.double() + 6.0).view(T, H, D)
    S, o = torch.zeros(H, D, Dv, dtype=torch.float64), torch.empty(T, H, Dv, dtype=torch.float64)
    for t in range(T):
        S = a[t][:, :, None] * S + k[t][:, :, None] * v[t][:, None]
        w = (S * q[t][:, :, None]).sum(1)
        o[t] = w / torch.sqrt((w * w).mean(-1, keepdim=True) + 1e-5)
    r = o.flatten(1) * torch.nn.functional.silu(gate)
    # differences of a running sum over eight tokens: 3e-7 to 5e-7
    assert _rel(y, r) < 2.5e-7
    assert _rel(st.S[0], S) < 2.5e-7


@pytest.mark.parametrize("spread", [8.0, 20.0])
def test_gates_that_close_hard(spread, monkeypatch):
    """As above for exponential gates, some of which forget almost everything."""
    from enterprise_inference_amd.ops import linear_scan as ls
    monkeypatch.setattr(ls, "FORCE_CHUNKED", True)
    H, D, T = 4, 64, 256
    g = torch.Generator().manual_seed(int(spread))
    x = torch.randn(T, 4 * H * D + 2 * H, generator=g)
    x[:, -H:] = 4 + spread * torch.randn(T, H, generator=g)
    at = [0, H * D, 2 * H * D, 3 * H * D, 4 * H * D, 4 * H * D + H]
    spec = ls.ScanSpec(H, D, D, "exp_gates", kscale=D ** -0.5, eps=1e-5, cap=0.0, gate_act="sigmoid")
    i32 = lambda v: torch.tensor(v, dtype=torch.int32, device="cuda")

    def run(x):
        st = ls.ScanState(torch.zeros(1, H, D, D, device="cuda"), torch.zeros(1, H, D, device="cuda"),
                          torch.zeros(1, H, device="cuda"))
        y = ls.linear_scan(x.cuda(), at[0], at[1], at[2], at[3], spec, st, i32([0]), i32([0, T]), 1,
                           torch.arange(T, dtype=torch.int32).cuda(), None, None, at[4], at[5],
                           plan=ls.chunk_plan([T], "cuda"))
        return y.cpu(), st.S[0].cpu()

    y, S = run(x)
    q, k, v, gate = (x[:, a:b].double() for a, b in zip(at, at[1:5]))
    q, k, v = q.view(T, H, D), k.view(T, H, D) * D ** -0.5, v.view(T, H, D)
    gi, gf = x[:, at[4]:at[5]].double(), torch.nn.functional.logsigmoid(x[:, at[5]:].double())
    s, n, m = (torch.zeros(*z, dtype=torch.float64) for z in ((H, D, D), (H, D), (H,)))
    o = torch.empty(T, H, D, dtype=torch.float64)
    for t in range(T):
        top = torch.maximum(gf[t] + m, gi[t])
        a, b, m = torch.exp(gf[t] + m - top), torch.exp(gi[t] - top), top
        s = a[:, None, None] * s + b[:, None, None] * k[t][:, :, None] * v[t][:, None]
        n = a[:, None] * n + b[:, None] * k[t]
        w = (s * q[t][:, :, None]).sum(1)
        w = w / (torch.maximum((n * q[t]).sum(-1).abs(), torch.exp(-m)) + 1e-6)[:, None]
        o[t] = w / torch.sqrt((w * w).mean(-1, keepdim=True) + 1e-5)
    # token by token 3e-7 and 5e-7; differences of two running sums over a block 3.5e-7 and 1e-6
    assert _rel(y, o.flatten(1) * torch.sigmoid(gate)) < 3e-7
    assert _rel(S, s) < 3e-7
    # a gate that is no number is not taken for one that closes
    for at_t in (5, 37, 130):
        bad = x.clone()
        bad[at_t, at[5] + 1] = float("nan")
        z, Z = run(bad)
        rest = [h for h in range(H) if h != 1]
        assert torch.equal(z[:at_t], y[:at_t]) and torch.isnan(z[at_t:, D:2 * D]).all() and torch.isnan(Z[1]).all()
        assert torch.equal(z.view(T, H, D)[:, rest], y.view(T, H, D)[:, rest]) and torch.equal(Z[rest], S[rest])


def test_linear_chunks_past_a_grid_column(monkeypatch):
    """More chunks than one dimension of the grid takes (chunk_grid: 32768): sequences of one token, whose output is
    (q . k) v / rms, and a longer one behind them, which comes out as it does alone."""
    from enterprise_inference_amd.ops import linear_scan as ls
    monkeypatch.setattr(ls, "FORCE_CHUNKED", True)
    lens, D = [1] * 32900 + [130], 16
    n, T = len(lens), sum(lens)
    g = torch.Generator().manual_seed(5)
    x = torch.randn(T, 64, generator=g).to(torch.bfloat16).cuda()
    cu = torch.tensor([0] + lens).cumsum(0).to(torch.int32).cuda()
    pos = torch.cat([torch.zeros(n - 1), torch.arange(130)]).to(torch.int32).cuda()
    spec = ls.ScanSpec(1, D, D, "decay", decay=torch.tensor([0.9]).cuda(), eps=1e-5)

    def run(x, cu, n, pos, lens):
        st = ls.ScanState.allocate(n, spec, "cuda")
        y = ls.linear_scan(x, 0, D, 2 * D, 3 * D, spec, st, torch.arange(n, dtype=torch.int32).cuda(), cu, n, pos,
                           plan=ls.chunk_plan(lens, "cuda"))
        return y, st.S

    y, S = run(x, cu, n, pos, lens)
    q, k, v, gate = x[:n - 1].float().split(D, 1)
    o = (q * k).sum(1, keepdim=True) * v
    want = o / torch.sqrt((o * o).mean(1, keepdim=True) + 1e-5) * torch.nn.functional.silu(gate)
    assert _rel(y[:n - 1], want) < 4e-3          # (one rounding to bf16 and at times one step more)
    assert _rel(S[:n - 1, 0], k[:, :, None] * v[:, None, :]) < 2e-6
    alone, Sa = run(x[n - 1:], torch.tensor([0, 130], dtype=torch.int32).cuda(), 1, pos[n - 1:], [130])
    assert torch.equal(y[n - 1:], alone) and torch.equal(S[n - 1:], Sa)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("mode,H,D,Dv", [("channel", 2, 64, 128), ("channel", 3, 32, 64), ("exp_gates", 2, 128, 128),
                                         ("decay", 2, 64, 64)])
def test_outputs_into_a_view(mode, H, D, Dv, dtype, monkeypatch):
    """Rows of an output that vector accesses cannot take hold the same numbers as rows that they can."""
    from enterprise_inference_amd.ops import linear_scan as ls
    monkeypatch.setattr(ls, "FORCE_CHUNKED", True)
    g = torch.Generator(device="cuda").manual_seed(D)
    lens = [130, 64, 1]
    T, n, W = sum(lens), len(lens), H * Dv
    at = [0, H * D, 2 * H * D, 2 * H * D + W, 2 * H * D + 2 * W, 2 * H * D + 2 * W + H]
    x = torch.randn(T, at[-1] + H + 8, generator=g, device="cuda").to(dtype)
    nw = (1 + 0.1 * torch.randn(W, generator=g, device="cuda")).to(dtype)
    spec = ls.ScanSpec(H, D, Dv, mode, kscale=D ** -0.5, eps=1e-5, decay=torch.linspace(0.9, 0.5, H).cuda(),
                       a2t=torch.randn(8, H * D, generator=g, device="cuda"), tau=8.0)
    cu, pos, slots = (t.cuda() for t in _step(lens, [0, 5, 0], False))

    def run(out, w):
        st = ls.ScanState.allocate(n, spec, "cuda")
        st.S.fill_(0.3)
        y = ls.linear_scan(x, at[0], at[1], at[2], at[3], spec, st, slots, cu, n, pos, None, w, at[4], at[5], out=out,
                           plan=ls.chunk_plan(lens, "cuda"), lo_off=at[-1] + H)
        return y.clone(), st.S

    y, S = run(None, nw)
    for left, width in ((3, W + 5), (4, W + 8)):
        z, R = run(torch.full((T, width), 7.0, device="cuda", dtype=dtype)[:, left:left + W], nw)
        assert torch.equal(z, y) and torch.equal(R, S)
    odd = torch.empty(W + 1, device="cuda", dtype=dtype)[1:].copy_(nw)
    assert torch.equal(run(None, odd)[0], y)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_wkv_rows_of_any_alignment(dtype):
    """Rows, weights and gates that vector accesses cannot take give what rows give that they can."""
    from enterprise_inference_amd.ops import wkv
    g = torch.Generator(device="cuda").manual_seed(3)
    lens, H, D = [130, 64, 300], 2, 64
    T, HD = sum(lens), H * D
    cu, pos, slots = (t.cuda() for t in _step(lens, [0, 5, 0], False))
    rnd = lambda *s: torch.randn(*s, generator=g, device="cuda")
    rows, dec, w0, u, nw = rnd(4, T, HD).to(dtype), rnd(T, HD), rnd(HD).to(dtype), rnd(HD).to(dtype), rnd(HD).to(dtype)
    x = rnd(T, 24)
    out = []
    for odd in (False, True):
        r, k, v, gate = rows
        w = nw
        if odd:
            r, k, v, gate = (torch.empty(T, HD + 3, device="cuda", dtype=dtype)[:, 1:1 + HD].copy_(t) for t in rows)
            w = torch.empty(HD + 1, device="cuda", dtype=dtype)[1:].copy_(nw)
        S = torch.full((3, H, D, D), 0.2, device="cuda")
        y = wkv.wkv_scan(r, k, v, gate, dec, w0, u, w, S, torch.zeros(3, 24, device="cuda"), x, slots, cu, 3, pos, None,
                         1e-5, H)
        out.append((y, S))
    # the same fp32 sums, whichever way their factors came
    assert _rel(out[1][0], out[0][0]) < (1e-6 if dtype == torch.float32 else 1e-3) and _rel(out[1][1], out[0][1]) < 1e-6


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("off,weight_off", [(0, 1), (4, 0), (4, 1), (2, 0)])
def test_wkv_rows_and_weights_aligned_apart(off, weight_off, dtype):
    """Rows that lie on 16 bytes beside weights that do not lie on four elements, and rows that do so the other way."""
    from enterprise_inference_amd.ops import wkv
    lens, H, D = [130, 64, 300], 2, 64
    T, HD = sum(lens), H * D
    cu, pos, slots = (t.cuda() for t in _step(lens, [0, 5, 0], False))
    args = [t.cuda() for t in _wkv_args(torch.Generator().manual_seed(off), T, 3, H, D, dtype)]
    S0, out = args[8].clone(), []
    for o, w in ((0, 0), (off, weight_off)):
        a = list(args)
        a[8] = S0.clone()
        a[:4] = (torch.empty(T, HD + 2 * o, device="cuda", dtype=dtype)[:, o:o + HD].copy_(t) for t in args[:4])
        a[7] = torch.empty(HD + w, device="cuda", dtype=dtype)[w:].copy_(args[7])
        out.append((wkv.wkv_scan(*a, slots, cu, 3, pos, None, 1e-5, H), a[8]))
    # the same fp32 sums, whichever way their factors came
    assert _rel(out[1][0], out[0][0]) < (1e-6 if dtype == torch.float32 else 1e-3) and _rel(out[1][1], out[0][1]) < 1e-6


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("Dv", [128, 64])
@pytest.mark.parametrize("off,weight_off,out_off", [(0, 1, 0), (0, 0, 2), (4, 0, 0), (4, 1, 4), (1, 0, 0)])
def test_channel_rows_and_weights_aligned_apart(off, weight_off, out_off, Dv, dtype, monkeypatch):
    """Rows that lie on 16 bytes beside weights or outputs that do not lie on four elements, and rows the other way."""
    from enterprise_inference_amd.ops import linear_scan as ls
    monkeypatch.setattr(ls, "FORCE_CHUNKED", True)
    lens, H, D, R = [130, 64, 200], 2, 64, 8
    T, W, at = sum(lens), H * Dv, [0, H * D, 2 * H * D, 2 * H * D + H * Dv, 2 * H * (D + Dv)]
    g = torch.Generator(device="cuda").manual_seed(Dv)
    rnd = lambda *s: torch.randn(*s, generator=g, device="cuda")
    rows, nw = rnd(T, at[-1] + R).to(dtype), (1 + 0.1 * rnd(W)).to(dtype)
    spec = ls.ScanSpec(H, D, Dv, "channel", kscale=D ** -0.5, eps=1e-5, a2t=rnd(R, H * D), tau=8.0)
    cu, pos, slots = (t.cuda() for t in _step(lens, [0, 5, 0], False))

    def run(o, w, b):
        x = torch.empty(T, rows.shape[1] + 2 * o, device="cuda", dtype=dtype)[:, o:o + rows.shape[1]].copy_(rows)
        weight = torch.empty(W + w, device="cuda", dtype=dtype)[w:].copy_(nw)
        out = torch.empty(T, W + b, device="cuda", dtype=dtype)[:, b:]
        st = ls.ScanState.allocate(3, spec, "cuda")
        st.S.fill_(0.3)
        y = ls.linear_scan(x, at[0], at[1], at[2], at[3], spec, st, slots, cu, 3, pos, None, weight, out=out,
                           plan=ls.chunk_plan(lens, "cuda"), lo_off=at[4])
        return y, st.S

    (y, S), (z, Z) = run(0, 0, 0), run(off, weight_off, out_off)
    # the same fp32 sums, whichever way their factors came
    assert _rel(z, y) < (1e-6 if dtype == torch.float32 else 1e-3) and _rel(Z, S) < 1e-6
