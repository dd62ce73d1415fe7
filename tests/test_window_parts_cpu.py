"""Workspaces of prefill launches in parts, against the register tiles of the kernels that write them."""

import pytest

from enterprise_inference_amd.ops import window_attention as wa


@pytest.mark.parametrize("maps,dim,vdim,tiles", [
    (2, 64, 128, 4), (2, 40, 48, 4), (2, 16, 16, 4),          # pairs: one kernel, four tiles
    (1, 16, 16, 2), (1, 32, 32, 2), (1, 64, 64, 2), (1, 40, 112, 4), (1, 72, 48, 3), (1, 96, 96, 3),
    (1, 96, 112, 4), (1, 128, 16, 4)])
@pytest.mark.parametrize("heads,kv_heads,queries", [(8, 2, 32), (3, 1, 128), (6, 3, 64)])
def test_flash_workspace(heads, kv_heads, queries, maps, dim, vdim, tiles):
    spec = wa.WindowSpec(heads, kv_heads, maps, dim, vdim, 0, 0, None)
    row_blocks, parts = 5 * heads * queries // 128, 3
    # four waves a map, each 16 sums a lane and tile, and four floats beside them
    assert wa.flash_workspace(5, spec, queries, parts) == row_blocks * parts * 4 * maps * 64 * (16 * tiles + 4)
