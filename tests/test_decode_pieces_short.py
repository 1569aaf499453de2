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


def _turns(live):
    """Turns of the waves of each record's block: four blocks of keys one turn, the entry's last part one more for the new key."""
    return -(-(live[:, 3] - live[:, 2]) // 4) + (live[:, 4] == live[:, 5] - 1)


@pytest.mark.parametrize("blocks", [9, 13, 19, 25, 33, 37, 41, 50, 64])
@pytest.mark.parametrize("requests", [1, 2, 4])
def test_finer_parts_take_no_turn_more_than_parts_of_eight(requests, blocks):
    """Parts of four blocks of 25 or 37 leave one over, which the last part would take as a third turn; and more than eight
    parts are more than the merging block asks for at a time."""
    rec = key_pieces.decode_pieces(np.full(requests, 32 * blocks), 8)
    live = rec[rec[:, 0] >= 0]
    eight = key_pieces._piece_sizes(np.array([blocks]), 8, True)[0][0]
    eight = eight[eight > 0]
    assert _turns(live).max() <= max(-(-eight[0] // 4), -(-eight[-1] // 4) + 1) and live[0, 5] <= 8 and len(live) <= key_pieces.PIECE_UNITS


@pytest.mark.parametrize("lengths", [(700,) * 8, (300,) * 12, (300,) * 16, (820, 1300, 1060, 340, 580, 100), (700, 400, 1000, 1300, 100)])
def test_more_requests_go_in_parts_of_eight_blocks_or_whole(lengths):
    """Parts of four blocks of these were up to an eighth slower: more pieces than compute units, more parts to merge."""
    rec = key_pieces.decode_pieces(np.array(lengths), 8)
    live = rec[rec[:, 0] >= 0]
    assert len(live) <= key_pieces.PIECE_UNITS and live[:, 5].max() <= 8


@pytest.mark.parametrize("requests", [1, 3, 4])
def test_the_choice_for_few_requests_counts_the_parts_that_are_cut(requests):
    rng = np.random.default_rng(requests)
    for _ in range(200):
        nblk = rng.integers(1, 65, requests)
        choice = key_pieces._few_width(nblk, 4)
        if choice:
            sizes, parts = key_pieces._piece_sizes(nblk, *choice)
            assert sizes.sum(axis=1).tolist() == nblk.tolist() and parts.max() <= 8 and parts.sum() * 4 <= key_pieces.PIECE_UNITS
