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
