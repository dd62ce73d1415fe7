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


# (row blocks, longest and mean tiles, slots, the merge's time in tiles): tiles per part that measured best, of the
# docstring's lists; within two tiles, or within one of the whole row block
@pytest.mark.parametrize("wgs,tiles,mean,slots,merge,best", [
    (220, 56, 28, 512, 6, 18), (314, 80, 40, 512, 6, 40), (344, 86, 44, 512, 6, 43), (376, 94, 48, 512, 6, 47),
    (400, 100, 50, 512, 6, 50), (420, 106, 54, 512, 6, 53), (422, 40, 21, 512, 6, 20), (436, 109, 55, 512, 6, 55),
    (438, 110, 55, 512, 6, 55), (438, 110, 56, 512, 6, 55), (500, 126, 64, 512, 6, 63), (504, 38, 20, 512, 6, 19),
    (512, 64, 32, 512, 6, 32), (454, 66, 34, 512, 6, 33),
    (324, 14, 8, 512, 6, 7), (408, 12, 7, 512, 6, 12), (410, 16, 11, 512, 6, 16), (456, 30, 18, 512, 6, 30),
    (348, 26, 16, 512, 6, 13), (412, 52, 27, 512, 6, 26),
    (688, 86, 44, 768, 7, 86), (752, 94, 48, 768, 7, 94), (512, 34, 18, 768, 7, 34), (326, 14, 8, 768, 7, 14),
    (488, 14, 8, 768, 7, 14), (540, 18, 10, 768, 7, 18), (410, 78, 47, 768, 7, 39), (338, 56, 29, 768, 7, 18),
    (166, 16, 12, 256, 3, 13), (160, 36, 30, 256, 3, 30), (152, 38, 19, 256, 3, 19), (186, 24, 13, 256, 3, 12),
    (233, 36, 19, 256, 3, 18), (185, 48, 36, 256, 3, 24), (410, 30, 16, 512, 11, 30), (462, 68, 39, 512, 11, 34)])
def test_parts_near_the_best_measured(wgs, tiles, mean, slots, merge, best):
    parts, per = split_keys(wgs, tiles, mean, slots, 12, merge)
    assert abs(per - best) <= (2 if best < tiles else 1)


@pytest.mark.parametrize("slots", [256, 512])
def test_no_part_is_longer_than_half_a_causal_row_block(slots):
    for wgs in range(1, slots + 1):
        for tiles in (50, 64, 110, 300):
            parts, per = split_keys(wgs, tiles, tiles // 2, slots)
            assert parts >= 2 and 2 * per <= tiles + 1


@pytest.mark.parametrize("merge", [3, 7, 11])
@pytest.mark.parametrize("slots", [256, 512, 768])
def test_parts_cover_every_tile_whatever_the_merge_takes(slots, merge):
    for wgs in (1, 127, 128, 129, 256, 257, 376, 512, 700, 768, 769):
        for tiles in (12, 13, 24, 65, 300):
            for mean in (tiles // 2, 3 * tiles // 4, tiles):
                parts, per = split_keys(wgs, tiles, mean, slots, 12, merge)
                assert per >= 1 and parts * per >= tiles > (parts - 1) * per
                assert parts == 1 or (wgs <= slots and per >= 6)
