"""The cut of a few requests' keys where a part has few blocks: every part a turn of its block's four waves or more, whole
entries where a cut saves no more than the parts' merge costs, and parts that still tile the entry's blocks."""
import numpy as np
import pytest

from spyinfer_amd.kernels import key_pieces


@pytest.mark.parametrize("blocks, parts", [(1, 1), (4, 1), (8, 1), (16, 4), (24, 6), (28, 7)])
@pytest.mark.parametrize("requests", [1, 2, 4])
def test_parts_of_a_few_requests(requests, blocks, parts):
    for kv_len in (32 * blocks - 31, 32 * blocks):
        rec = key_pieces.decode_pieces(np.full(requests, kv_len), 8)
        live = rec[rec[:, 0] >= 0]
        assert (live[:, 5] == parts).all() and len(live) == requests * 8 * parts
        sizes = live[:, 3] - live[:, 2]
        assert sizes.sum() == requests * 8 * blocks and sizes.max() <= max(blocks if parts == 1 else 0, key_pieces.PIECE_MIN_BLOCKS)


@pytest.mark.parametrize("lengths", [(1, 33, 500, 4096), (129, 130), (38000,), (700, 20, 20, 20, 20)])
@pytest.mark.parametrize("n_kv, window, d", [(1, 0, 128), (8, 0, 64), (3, 200, 128)])
def test_parts_tile_the_keys(lengths, n_kv, window, d):
    rec = key_pieces.decode_pieces(np.array(lengths), n_kv, window, head_dim=d)
    live = rec[rec[:, 0] >= 0]
    for s, kv_len in enumerate(lengths):
        lo = (max(0, kv_len - window) if window else 0) & ~31
        for hk in range(n_kv):
            mine = live[(live[:, 0] == s) & (live[:, 1] == hk)]
            mine = mine[np.argsort(mine[:, 4])]
            assert len(mine) <= key_pieces.MAX_PARTS and (mine[:, 3] > mine[:, 2]).all()
            assert mine[0, 2] == 0 and mine[-1, 3] == (kv_len - 1 - lo) // 32 + 1 and (mine[1:, 2] == mine[:-1, 3]).all()
