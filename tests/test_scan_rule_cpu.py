"""Which form of a linear recurrence a step takes: both sides of the lines, at the sizes timed for them."""

import pytest

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
