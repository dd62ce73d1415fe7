"""How prefill launches cut their row blocks along the keys."""

import pytest

from enterprise_inference_amd.ops.attention import split_keys


@pytest.mark.parametrize("slots,least", [(256, 24), (512, 12), (768, 12)])
@pytest.mark.parametrize("tiles", [1, 11, 12, 13, 24, 64, 129, 1000])
@pytest.mark.parametrize("past", [0.0, 0.5, 0.9, 1.0])
def test_parts_cover_every_tile(slots, least, tiles, past):
    for wgs in (1, 2, 5, 64, 127, 128, 171, 255, 256, 257, 376, 511, 512, 513, 768, 769, 5000):
        mean = max(1, int(tiles * (1 + past) / 2))
        parts, per = split_keys(wgs, tiles, mean, slots, least)
        assert parts >= 1 and per >= 1 and parts * per >= tiles > (parts - 1) * per
        if wgs > slots or tiles < least:
            assert parts == 1
        if parts > 1:
            assert per >= least // 2
            # in one round, or two: of row blocks that grow to `tiles` a part each and half of one more
            assert wgs * min(parts, mean / per + 0.5) <= 2 * slots


def test_one_round_where_it_fits():
    assert split_keys(256, 64, 32, 512) == (3, 24)         # 480 parts on 512 slots
    assert split_keys(128, 18, 18, 512) == (3, 6)          # equally long: four parts would be under half of least
    assert split_keys(200, 18, 18, 512) == (1, 18)         # ... two parts of each do not pay
    assert split_keys(513, 64, 32, 512) == (1, 64)


@pytest.mark.parametrize("wgs,tiles,mean,best", [(220, 56, 28, 18), (314, 80, 40, 40), (344, 86, 44, 43), (376, 94, 48, 47),
                                                 (400, 100, 50, 50), (420, 106, 54, 53), (422, 40, 21, 20),
                                                 (436, 109, 55, 55), (438, 110, 55, 55), (438, 110, 56, 34), (482, 122, 62, 42)])
def test_parts_near_the_best_measured(wgs, tiles, mean, best):
    """Tiles per part of causal row blocks on 512 slots: the setting that measured best of the docstring's lists (438
    row blocks take halves or two rounds, which measured the same), within two tiles."""
    parts, per = split_keys(wgs, tiles, mean, 512)
    assert abs(per - best) <= 2


@pytest.mark.parametrize("slots", [256, 512])
def test_no_part_is_longer_than_half_a_row_block(slots):
    for wgs in range(1, slots + 1):
        for tiles in (24, 50, 64, 110, 300):
            parts, per = split_keys(wgs, tiles, tiles // 2, slots)
            assert parts >= 2 and 2 * per <= tiles + 1


def test_three_workgroups_on_a_cu():
    """... take no second round: 688 and 752 row blocks of heads of 64 measured best uncut."""
    assert split_keys(688, 86, 44, 768, crowded=True) == (1, 86)
    assert split_keys(752, 94, 48, 768, crowded=True) == (1, 94)
    for wgs in range(1, 769):
        parts, per = split_keys(wgs, 94, 47, 768, crowded=True)
        assert parts * per >= 94 > (parts - 1) * per and (parts == 1 or wgs * (47 / per + 0.5) <= 768)
