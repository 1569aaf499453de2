"""The cut of keys for blocks of eight waves: one block a compute unit at most, parts that tile the entries, and which steps have such blocks."""
import numpy as np
import pytest

from spyinfer_amd.kernels import key_pieces


def test_steps_with_blocks_of_eight_waves():
    assert [key_pieces.piece_waves(n, 8, 128) for n in (1, 20, 21, 64)] == [8, 8, 4, 4]
    assert key_pieces.piece_waves(1, 8, 64) == 4 and key_pieces.piece_waves(80, 2, 128) == 8 and key_pieces.piece_waves(81, 2, 128) == 4


@pytest.mark.parametrize("n_kv", [1, 2, 8, 32])
def test_every_piece_finds_a_unit(n_kv):
    rng = np.random.default_rng(n_kv)
    for _ in range(150):
        S = int(rng.integers(1, max(2, 5 * 256 // 8 // n_kv + 1)))
        kv_len = rng.integers(1, int(rng.choice([40, 600, 2000, 20000])), S)
        assert key_pieces.piece_waves(S, n_kv, 128) == 8
        rec = key_pieces.decode_pieces(kv_len, n_kv)
        live = rec[rec[:, 0] >= 0]
        assert len(live) <= key_pieces.PIECE_UNITS and live[:, 5].max() <= key_pieces.MAX_PARTS
        for s in range(S):
            mine = live[(live[:, 0] == s) & (live[:, 1] == 0)]
            mine = mine[np.argsort(mine[:, 4])]
            assert mine[0, 2] == 0 and mine[-1, 3] == (kv_len[s] - 1) // 32 + 1 and (mine[1:, 2] == mine[:-1, 3]).all()


def test_the_last_part_has_the_new_key():
    """What the kernel goes by: the part with the number parts - 1 ends where the entry does."""
    rec = key_pieces.decode_pieces(np.array([33, 700, 2, 1025, 64]), 8)
    live = rec[rec[:, 0] >= 0]
    last = live[live[:, 4] == live[:, 5] - 1]
    assert len(last) == 5 * 8 and (last[:, 3] == (last[:, 7] - 1) // 32 + 1).all()
