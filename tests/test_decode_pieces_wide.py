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


def test_more_entries_than_half_of_the_units_have_such_blocks_for_few_keys_only():
    """17 to 20 entries of 8 kv heads leave 96 to 120 units of 256 for the parts of 136 to 160 whole entries: with many keys the longest stay whole, and the
    step waits for them."""
    waves = key_pieces.piece_waves
    assert [waves(n, 8, 128, 1024) for n in (16, 17, 20, 21)] == [8, 8, 8, 4] and [waves(n, 8, 128, 1025) for n in (1, 16, 17, 20)] == [8, 8, 4, 4]
    assert waves(64, 2, 128, 5000) == 8 and waves(65, 2, 128, 5000) == 4
    assert key_pieces.keys_read(5000, 0) == 5000 and key_pieces.keys_read(5000, 512) == 543 and key_pieces.keys_read(100, 512) == 100


@pytest.mark.parametrize("lens,window,waves", [([2500] * 20, 0, 4), ([250 + 118 * i for i in range(20)], 0, 4), ([700] * 20, 0, 8), ([2500] * 20, 512, 8), ([2500] * 16, 0, 8)])
def test_the_plan_of_a_step_says_which_blocks_it_is_cut_for(lens, window, waves):
    from spyinfer_amd.parts import attention

    class Batch:
        S, lens_, max_kv_len, shared, arrays, keys = len(lens), lens, max(lens), {}, {}, {}
        host_array = staticmethod(lambda name: np.array(lens))
        add_array = staticmethod(lambda name, values: Batch.arrays.__setitem__(name, values))
        add_graph_key = staticmethod(lambda name, value: Batch.keys.__setitem__(name, value))

    attention.plan_decode_pieces(Batch, 8, window, 128)
    assert list(Batch.keys.values()) == [waves]                      # (a launch shape: steps with other blocks are other graphs)
    rec = next(iter(Batch.arrays.values()))
    live = rec[rec[:, 0] >= 0]
    assert (len(live) <= key_pieces.PIECE_UNITS) == (waves == 8)
    # the unit with most blocks of keys, of all that it has in two rounds, against an even share
    sizes = live[:, 3] - live[:, 2]
    load = np.zeros(key_pieces.PIECE_UNITS)
    load[:min(len(sizes), 256)] += sizes[:256]
    load[:max(0, len(sizes) - 256)] += sizes[256:]
    assert waves == 8 or load.max() <= 1.35 * sizes.sum() / key_pieces.PIECE_UNITS


@pytest.mark.parametrize("requests", [1, 2, 4])
@pytest.mark.parametrize("blocks", [29, 37, 45, 55])
def test_few_requests_are_cut_for_the_blocks_that_they_get(requests, blocks):
    """Blocks of eight waves, whose time goes by their blocks of keys: eight parts, not as many as blocks of four waves have turns (29 blocks, microseconds:
    six parts 10.0, eight 9.6; 37: 11.3, 11.0; 45: 11.6, 11.4)."""
    rec = key_pieces.decode_pieces(np.full(requests, 32 * blocks), 8)
    live = rec[rec[:, 0] >= 0]
    assert (live[:, 5] == 8).all()


def test_the_cut_of_a_step_follows_its_lengths_without_being_kept():
    """Nothing is kept by all of a step's lengths: with uneven ones these are new in almost every step."""
    rng = np.random.default_rng(4)
    lens = rng.integers(50, 1300, 16)
    key_pieces._piece_choices.clear()
    for step in range(64):
        key_pieces.decode_pieces(lens + step, 8)
    assert not key_pieces._piece_choices
    # the first width, by the longest entry's estimated time, that gives every piece a unit: as looking at every width finds it
    for _ in range(200):
        n_kv = int(rng.integers(1, 9))
        nblk = rng.integers(1, 200, int(rng.integers(1, 160 // n_kv + 1)))
        choice = key_pieces._wide_width(nblk, n_kv)
        order = key_pieces._wide_order(int(nblk.max()), 4, key_pieces.PIECE_MERGE_US, key_pieces.PIECE_MERGE_MORE_US, nblk.shape[0] <= key_pieces.PIECE_FEW)
        fits = [w for w, _ in order if int((-(-nblk // w)).sum()) * n_kv <= key_pieces.PIECE_UNITS]
        assert (fits[0] if -(-int(nblk.max()) // fits[0]) > 1 else None) == (choice and choice[0])
