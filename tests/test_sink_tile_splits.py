"""How many workgroups share a tile's keys follows the tiles of a step, not its rows alone."""
import pytest

from swifttransformer_amd.ops import kernels as K


@pytest.mark.parametrize("heads,kv_heads,dim,mixed,slots", [(32, 8, 64, True, 256), (32, 8, 64, False, 256), (16, 2, 128, False, 256), (6, 2, 64, False, 256)])
def test_single_tokens_are_tiles_too(heads, kv_heads, dim, mixed, slots):
    splits = lambda rows, items: K.sink_tile_splits(rows, items, heads, kv_heads, dim, dim, mixed, 1024)
    assert splits(128, 1) == 8                                 # nine tiles at most: the limit
    assert splits(128, 101) <= 3                               # 100 single tokens and a portion of 28
    assert splits(512, 300) == 1 and splits(4096, 1) == 1
    for rows, items in ((128, 1), (128, 65), (256, 65), (512, 3), (2048, 1), (1000, 40)):
        tiles = rows // 16 + items
        # no more than half again of the workgroups that the chip holds
        assert splits(rows, items) == 1 or splits(rows, items) * tiles <= 1.5 * slots
    assert K.sink_tile_splits(128, 1, heads, kv_heads, dim, dim, mixed, 255) == 1      # at least 128 keys a share
