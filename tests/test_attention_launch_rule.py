"""The rule that sends a step's large and small attention tiles through one launch or two, asked about steps that were measured (where
the two ways differ by more than 4 %), and the numbers of keys that the plan hands it."""
import numpy as np
import pytest

from spyinfer_amd.kernels import ops
from spyinfer_amd.parts import attention

# n_q, n_kv, d, (cached, new) of the entries with large tiles, (how many, fewest keys, most keys) of the single tokens beside them, together?
MEASURED = [
    (32, 8, 128, [(0, 389)], (20, 60, 700), True),             # 38.3 us apart, 24.2 together
    (32, 8, 128, [(0, 389)], (96, 300, 500), True),            # 60.1 / 45.5
    (32, 8, 128, [(0, 389)], (96, 60, 1000), True),            # 79.4 / 58.3
    (32, 8, 128, [(0, 100)], (32, 1400, 1400), True),          # 46.6 / 40.4
    (32, 8, 128, [(0, 1000)], (96, 20, 60), True),             # 53.1 / 42.0
    (16, 8, 128, [(0, 1000)], (200, 100, 240), True),          # 71.7 / 61.6
    (32, 8, 128, [(0, 64)], (200, 100, 240), False),           # 49.2 / 53.6
    (32, 8, 128, [(0, 389)], (256, 200, 200), False),          # 67.7 / 75.1
    (32, 8, 128, [(0, 389)], (400, 300, 300), False),          # 111.2 / 129.2
    (16, 8, 128, [(0, 64)], (400, 50, 150), False),            # 63.7 / 80.1
    (32, 8, 128, [(0, 1000), (0, 900)], (64, 1000, 1000), False),   # 92.8 / 100.0
    (32, 8, 128, [(0, 60)] * 30, (96, 1000, 1000), False),     # 90.0 / 103.8
    (32, 8, 128, [(0, 2000)], (96, 1000, 1000), False),        # 139.3 / 152.8
    (32, 8, 128, [(0, 100)], (1, 8000, 8000), False),          # 30.4 / 98.7
    (32, 8, 64, [(0, 389)], (400, 300, 300), True),            # 69.7 / 56.0
    (32, 8, 64, [(0, 64)], (128, 1000, 1000), True),           # 57.4 / 48.0
]


class Batch:
    """What plan_attention_tiles reads of a step."""

    def __init__(self, entries):
        self.S, self.lens = len(entries), np.array([n for _, n in entries], dtype=np.int32)
        self.host = dict(pos0=np.array([a for a, _ in entries], dtype=np.int32), kv_len=np.array([a + n for a, n in entries], dtype=np.int32))
        self.max_kv_len, self.shared, self.arrays = int(self.host["kv_len"].max()), {}, {}

    def host_array(self, name):
        return self.host[name]

    def add_array(self, name, values):
        self.arrays[name] = values

    def add_graph_key(self, name, value):
        pass


def planned(entries, group, chunk=0):
    batch = Batch(entries)
    attention.plan_attention_tiles(batch, group, 128, chunk=chunk)
    return batch, batch.shared.get(("attention_keys", group, 128, chunk))


@pytest.mark.parametrize("n_q, n_kv, d, large, small, together", MEASURED)
def test_the_way_that_was_faster(n_q, n_kv, d, large, small, together):
    n, lo, hi = small
    batch, keys = planned(large + [(int(k), 1) for k in np.linspace(lo, hi, n).astype(int)], n_q // n_kv)
    tiles = batch.shared[("attention_tiles", n_q // n_kv, 128, 0)]
    assert ops.mixed_attention_pays(tiles["big"] * n_kv, keys["max_big_keys"], keys["max_small_keys"], d, tiles["small"] * n_kv,
                                    keys["big_keys"] * n_kv, keys["small_keys"] * n_kv) == together


def test_the_plan_counts_the_keys_that_the_tiles_read():
    _, keys = planned([(10, 40), (0, 100), (500, 1), (20, 6), (0, 5)], 4)
    # 128-row tiles hold 32 tokens: 10 + 32 and all 50 keys, then 32, 64, 96 and 100; 16-row tiles four tokens, each reading the entry's keys
    assert keys == dict(max_big_keys=100, max_small_keys=501, big_keys=42 + 50 + 32 + 64 + 96 + 100, small_keys=501 + 2 * 26 + 2 * 5)
    assert planned([(0, 50), (3, 1)], 4)[1] == dict(max_big_keys=50, max_small_keys=4, big_keys=32 + 50, small_keys=4)
    # in chunks of 48 positions the keys of a tile start at its first row's chunk
    assert planned([(40, 40), (3, 1)], 4, chunk=48)[1]["big_keys"] == 72 + (80 - 48)
    # a step without large tiles has nothing to choose
    assert planned([(30, 1), (3, 1)], 4)[1] is None


# d, (128-row tiles, kv heads), the most keys of an entry, parts: the fastest measured, or within 2 % of it and of the most parts
PARTS = [(128, 16, 8, 512, 1), (128, 32, 8, 1000, 1), (128, 10, 8, 1300, 3), (128, 4, 8, 2100, 6), (128, 13, 8, 2400, 4), (128, 7, 8, 4200, 6),
         (64, 5, 8, 1300, 5), (64, 7, 8, 4200, 9), (64, 3, 8, 8064, 16), (64, 8, 8, 512, 1), (128, 4, 8, 64, 1)]


@pytest.mark.parametrize("d, tiles, n_kv, keys, parts", PARTS)
def test_parts_of_the_keys_of_few_large_tiles(d, tiles, n_kv, keys, parts):
    assert ops.prefill_key_parts(tiles * n_kv, keys, d) == parts
