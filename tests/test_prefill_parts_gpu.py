"""Flash prefill whose query blocks are cut along the keys: parts of one tile, parts that do not divide a block's
tiles, more tiles than the parts were counted for, waves without queries and parts without keys."""

import pytest
import torch

BF = torch.bfloat16


def test_parts_cover_and_fit():
    from enterprise_inference_amd.ops.attention import FA_SLOTS, fa_parts
    for wgs in (1, 2, 7, 16, 40, 64, 127, 128, 129, 192, 232, 255, 256, 257, 4000):
        for tiles in (1, 2, 5, 6, 16, 33, 64, 500, 2049, 40000):
            for share in (0.5, 0.6, 0.75, 0.9, 1.0):
                parts, per = fa_parts(wgs, tiles, max(1.0, tiles * share))
                assert parts >= 1 and 1 <= per <= tiles and (parts - 1) * per < tiles <= parts * per
                assert parts == 1 or (wgs <= FA_SLOTS and wgs * parts <= 1024)


@pytest.mark.parametrize("KT,two", [(64, True), (64, False), (32, False)])
@pytest.mark.parametrize("lens,past", [([1], 0), ([9], 1000), ([200, 31], 0), ([500, 3, 90], 5000)])
@pytest.mark.parametrize("window", [0, 300])
def test_latent_parts_cover(lens, past, window, KT, two):
    from enterprise_inference_amd.ops.latent_attention import flash_parts
    context = -(-(past + max(lens)) // 128) * 128
    tiles = -(-context // KT) if window == 0 else min(-(-context // KT), window // KT + 2)
    for wgs in (1, 13, 64, 65, 128, 157, 256, 257, 600):
        parts, per = flash_parts(wgs, lens, context, tiles, KT, window, two)
        assert per >= 1 and parts * per >= tiles > (parts - 1) * per
        assert parts == 1 or wgs * parts <= max(1024, 3 * 512)


# (workgroups, longest and mean tiles, us a tile), times in us by tiles per part and uncut (0), of fa_parts' lists and
# of launches that a cut made slower
@pytest.mark.parametrize("launch,us", [
    ((56, 8, 4.8, 1.65), {0: 16.3, 2: 19.5, 3: 18.1, 4: 17.6}), ((42, 8, 4.8, 1.65), {0: 16.2, 3: 17.0}),
    ((200, 26, 13.9, 1.65), {0: 45.5, 22: 46.3, 13: 39.8}), ((192, 30, 18.1, 1.65), {0: 52.4, 15: 51.4, 26: 53.3}),
    ((192, 40, 25.0, 1.95), {0: 78.1, 12: 79.1, 20: 75.2}), ((168, 12, 6.0, 1.95), {0: 30.5, 7: 35.5}),
    ((112, 10, 6.3, 1.95), {0: 25.5, 5: 26.1}), ((192, 28, 16.1, 1.65), {0: 51.5, 23: 58.2}),
    ((24, 34, 33.4, 1.65), {0: 59.0, 5: 21.3, 9: 25.2}), ((120, 16, 8.6, 1.65), {0: 30.6, 6: 24.3}),
    ((128, 18, 10.1, 1.65), {0: 35.4, 8: 27.6}), ((128, 78, 70.2, 1.65), {0: 131, 39: 88.4}),
    ((52, 28, 26.1, 1.65), {0: 48.4, 7: 26.5}), ((120, 32, 17.4, 1.65), {0: 57.3, 13: 35.8}),
    ((164, 44, 23.6, 1.65), {0: 76.8, 26: 57.5}), ((112, 16, 8.7, 1.95), {0: 33.8, 6: 26.1}),
    ((236, 60, 30.5, 1.65), {0: 104.5, 19: 102.3, 30: 87.0}), ((208, 52, 26.4, 1.65), {0: 88.9, 14: 78.8, 26: 71.2}),
    ((104, 26, 13.1, 1.65), {0: 47.2, 8: 29.5}), ((192, 36, 35.5, 1.95), {0: 55.5, 18: 66.1})])
def test_a_cut_is_not_slower(launch, us):
    """Parts are of a length that was measured, and was not slower than the uncut launch."""
    from enterprise_inference_amd.ops.attention import fa_parts
    parts, per = fa_parts(*launch)
    assert us[0 if parts == 1 else per] <= us[0]
    assert parts > 1 or min(us.values()) > 0.85 * us[0]


# times in us by tiles per part, as measured, and the one that split_keys' rule took
@pytest.mark.parametrize("wgs,lens,context,tiles,KT,window,us,most", [
    (55, [871], 896, 14, 64, 1024, {2: 50.6, 3: 35.6, 4: 36.8, 6: 43.9, 14: 65.8}, 43.9),
    (56, [891], 896, 14, 64, 0, {2: 51.7, 3: 35.6, 4: 36.9, 6: 42.6, 14: 66.1}, 42.6),
    (26, [108, 90, 80, 100], 1472, 18, 64, 1024, {2: 54.3, 3: 34.5, 4: 36.7, 6: 42.0}, 42.0),
    (128, [261, 230, 190, 180, 140], 384, 6, 64, 1024, {2: 27.8, 3: 29.5, 6: 27.3}, 27.3),
    (41, [162], 768, 24, 32, 0, {4: 61.9, 5: 41.0, 6: 42.0, 12: 58.6}, 58.6)])
def test_latent_cuts_are_not_slower(wgs, lens, context, tiles, KT, window, us, most):
    """The parts of a workgroup run on one XCD: 26 of nine parts are 36 on some, which run 32 at a time."""
    from enterprise_inference_amd.ops.latent_attention import flash_parts
    assert us[flash_parts(wgs, lens, context, tiles, KT, window, False)[1]] <= most


def test_short_window_launches_are_not_cut():
    """Up to 6 tiles, us uncut and in parts of two: 14.0 / 15.9, 16.5 / 18.0, 16.1 / 17.0."""
    from enterprise_inference_amd.ops import window_attention as wa
    spec = lambda heads, kv, maps, dim, vdim, window: wa.WindowSpec(heads, kv, maps, dim, vdim, window, 0, None)
    assert wa.flash_parts(11, spec(16, 4, 1, 96, 96, 0), 32, 328, 384) == (1, 6)
    assert wa.pair_parts(16, spec(8, 2, 2, 64, 128, 1024), 32, 384) == (1, 6)
    assert wa.flash_parts(16, spec(8, 2, 1, 128, 128, 1024), 32, 260, 384) == (1, 6)


def test_launches_without_work_are_not_cut():
    from enterprise_inference_amd.ops import latent_attention as la
    from enterprise_inference_amd.ops import window_attention as wa
    from enterprise_inference_amd.ops.attention import fa_parts
    spec = wa.WindowSpec(8, 2, 1, 128, 128, 0, 0, mult=None)
    assert fa_parts(0, 32, 32.0) == wa.pair_parts(0, spec, 64, 2048) == wa.flash_parts(0, spec, 64, 1, 2048) == (1, 32)
    for lens in ([1], [0], [0, 0]):
        assert la.flash_parts(0, lens, 2048, 32, 64, 0, True) == (1, 32)


@pytest.mark.gpu
@pytest.mark.parametrize("cu", [[0], [0, 0]])
def test_flash_prefill_without_work(cu):
    """No sequences, and one without tokens, beside a block table of many pages."""
    from enterprise_inference_amd.ops import attention
    i32 = lambda *v: torch.tensor(v, dtype=torch.int32, device="cuda")
    q = torch.empty(0, 8, 128, dtype=BF, device="cuda")
    k, v = torch.zeros(1, 2, 128, 128, dtype=BF, device="cuda"), torch.zeros(1, 2, 128, 128, dtype=BF, device="cuda")
    bt, sl = torch.zeros(len(cu) - 1, 16, dtype=torch.int32, device="cuda"), i32(*[0] * (len(cu) - 1))
    assert attention.paged_prefill(q, k, v, bt, sl, i32(*cu), i32(), 0, 0.1).shape == q.shape


@pytest.mark.gpu
@pytest.mark.parametrize("Hq,Hkv", [(8, 2), (6, 3), (3, 1)])
@pytest.mark.parametrize("qlens,ctxs", [([1, 33, 64, 127], [700, 5, 70, 0]), ([255, 40], [63, 600]), ([300], [0])])
@pytest.mark.parametrize("causal,window,chunk", [(True, None, None), (False, None, None),
                                                 (True, 200, None), (True, None, 192)])
@pytest.mark.parametrize("parts,per", [(12, 1), (5, 3), (3, 2)])
def test_flash_prefill_parts(Hq, Hkv, qlens, ctxs, causal, window, chunk, parts, per, monkeypatch):
    from enterprise_inference_amd.ops import attention
    from enterprise_inference_amd.ops import reference as ref
    g = torch.Generator().manual_seed(sum(qlens) + Hq)
    D, bs = 128, 128
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
    q[0] = 0                                               # (equal scores)
    sl = torch.tensor(lens, dtype=torch.int32)
    cu = torch.tensor([0] + qlens).cumsum(0).to(torch.int32)
    r = ref.paged_attention_prefill(q.float(), k.float(), v.float(), bt, cu, sl, D ** -0.5, causal,
                                    window, chunk)
    work = torch.tensor(attention.build_prefill_work(
        qlens, attention.prefill_query_block(Hq, Hkv, D, block_size=bs)), dtype=torch.int32)
    asked = []
    monkeypatch.setattr(attention, "fa_parts", lambda *a: asked.append(a) or (parts, per))
    d = [t.cuda() for t in (q, k, v, bt, sl, cu, work)]
    o = attention.paged_prefill(*d[:6], d[6], work.numel() // 2, D ** -0.5, causal, window, chunk)
    assert asked                                           # (it was cut)
    # weights and outputs rounded to bf16 (2^-9 each, relative), fp32 sums
    err = (o.double().cpu() - r.double()).norm() / r.double().norm()
    assert err < 4e-3


@pytest.mark.gpu
@pytest.mark.parametrize("Hq,Hkv,qlens,ctxs", [(24, 8, [300, 40], [0, 500]), (16, 4, [640, 90], [300, 5]), (4, 1, [1500], [100])])
@pytest.mark.parametrize("parts,per", [(12, 1), (15, 1)])
def test_flash_prefill_parts_of_several_rounds(Hq, Hkv, qlens, ctxs, parts, per, monkeypatch):
    """More than 256 parts: those of a block do not stand together in the grid."""
    from enterprise_inference_amd.ops import attention as a
    blocks = sum(-(-n // a.prefill_query_block(Hq, Hkv, 128, block_size=128)) for n in qlens)
    assert blocks * (Hq // a.heads_per_workgroup(Hq, Hkv)) * parts > 256
    test_flash_prefill_parts(Hq, Hkv, qlens, ctxs, True, None, None, parts, per, monkeypatch)


@pytest.mark.gpu
def test_flash_prefill_counts_the_keys_behind_a_query(monkeypatch):
    """Without a causal mask a window does not bound what a block walks."""
    from enterprise_inference_amd.ops import attention
    asked = []
    monkeypatch.setattr(attention, "fa_parts", lambda *a: asked.append(a) or (1, a[1]))
    i32 = lambda *v: torch.tensor(v, dtype=torch.int32, device="cuda")
    q = torch.zeros(64, 8, 128, dtype=BF, device="cuda")
    k, v = torch.zeros(16, 2, 128, 128, dtype=BF, device="cuda"), torch.zeros(16, 2, 128, 128, dtype=BF, device="cuda")
    bt = torch.arange(16, dtype=torch.int32, device="cuda")[None]
    for causal, tiles in ((True, 6), (False, 32)):
        attention.paged_prefill(q, k, v, bt, i32(2048), i32(0, 64), i32(0, 0), 1, 0.1, causal, 200)
        assert asked[-1][1] == tiles
