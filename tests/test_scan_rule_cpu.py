"""Which form of a linear recurrence a step takes: both sides of the lines, at the sizes timed for them."""

import pytest

from enterprise_inference_amd.ops import wkv
from enterprise_inference_amd.ops.linear_scan import ChunkPlan


@pytest.mark.parametrize("mode,heads,dim,key_dim,nseq,rows,chunks", [
    ("decay", 32, 64, 64, 16, 64, False), ("decay", 32, 64, 64, 16, 128, True), ("decay", 32, 64, 64, 64, 64, False),
    ("decay", 16, 128, 128, 16, 64, False), ("decay", 16, 128, 128, 16, 128, True), ("decay", 16, 128, 128, 1, 4096, True),
    ("exp_gates", 32, 64, 64, 16, 48, False), ("exp_gates", 32, 64, 64, 64, 64, True),
    ("exp_gates", 16, 128, 128, 16, 48, True), ("exp_gates", 16, 128, 128, 64, 64, True),
    ("channel", 32, 64, 32, 16, 96, False), ("channel", 32, 64, 32, 16, 128, True),
    ("channel", 16, 128, 64, 64, 64, True), ("channel", 16, 128, 128, 16, 8, False)])
def test_pays(mode, heads, dim, key_dim, nseq, rows, chunks):
    plan = ChunkPlan([rows] * nseq, "cpu", 32)
    assert plan.pays(heads, dim, channel=mode == "channel", key_dim=key_dim, exp_gates=mode == "exp_gates") == chunks


@pytest.mark.parametrize("lens,heads,not_told,told", [
    ([200], 32, 1, 1), ([40], 32, 0, 0),
    # none is long: they stay token by token unless they all are nearly as long
    ([32] * 16, 32, 64, 0), ([24] * 8, 32, 56, 0), ([20] * 16, 16, 56, 0), ([40, 20] * 8, 16, 56, 0), ([50] * 8, 32, 12, 0),
    # one is
    ([500] + [24] * 15, 16, 12, 12), ([500] + [24] * 63, 16, 80, 51), ([160] + [20] * 15, 32, 64, 25),
    ([1, 300], 16, 1, 1), ([300, 300], 64, 6, 6)])
def test_wkv_rows_in_chunks(lens, heads, not_told, told):
    assert wkv.chunk_split(sum(lens), len(lens), heads) == not_told
    assert wkv.chunk_split(sum(lens), len(lens), heads, max(lens)) == told
