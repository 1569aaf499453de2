"""The sizes that go to blocks of more than eight row tiles, and what these are launched with: within what the kernel takes, for every size."""
import random

from spyinfer_amd.kernels import ops


def test_launches_fit_the_kernel():
    rng = random.Random(7)
    taken = 0
    for _ in range(6000):
        M, N, K = int(2 ** rng.uniform(5, 14)), 16 * rng.randint(1, 2000), 128 * rng.randint(1, 120)
        for kind in (ops.ROWS_STORE, ops.ROWS_PARTS, ops.ROWS_GATED):
            other = ops.rows_product_gated.__wrapped__(M, N, K, True) if kind == ops.ROWS_GATED and N % 32 == 0 else 0
            plan = ops.rows_product_tall.__wrapped__(M, N, K, kind, other)
            if plan is None:
                continue
            taken += 1
            tiles, parts = plan
            rows = -(-M // 16)
            assert 9 <= tiles <= 16 and 16 * tiles <= M and N * K < 1 << 30 and M * K < 1 << 30 and N % (32 if kind == ops.ROWS_GATED else 16) == 0
            shared = -(-rows // tiles)                       # (as the launcher deals them)
            assert -(-rows // shared) == tiles and shared * tiles * 16 >= M
            assert parts == 1 or kind == ops.ROWS_PARTS and parts <= K // 512 and parts * M * N * 4 <= ops.PARTS_MAX_BYTES
    assert taken > 300


def test_sizes_on_both_sides_of_the_line():
    tall = lambda *size: ops.rows_product_tall(*size) is not None
    assert tall(409, 19456, 2560, ops.ROWS_GATED, 6) and not tall(360, 19456, 2560, ops.ROWS_GATED, 8) and not tall(640, 12288, 2048, ops.ROWS_GATED, 8)
    assert tall(300, 24576, 4096, ops.ROWS_GATED) and tall(2048, 24576, 4096, ops.ROWS_GATED) and not tall(550, 24576, 4096, ops.ROWS_GATED, 7)
    assert tall(2048, 6144, 4096, ops.ROWS_STORE) and not tall(900, 6144, 4096, ops.ROWS_STORE) and not tall(2048, 8192, 2048, ops.ROWS_STORE)
    assert ops.rows_product_tall(2048, 4096, 12288, ops.ROWS_PARTS) == (16, 2) and not tall(640, 2560, 9728, ops.ROWS_PARTS)
    assert not tall(1500, 4096, 4096, ops.ROWS_PARTS) and tall(640, 4096, 4096, ops.ROWS_PARTS) and not tall(128, 24576, 4096, ops.ROWS_GATED)


def test_estimates_are_near_what_was_measured():
    """Microseconds of launches with another matrix each, from memory; both estimates within a tenth (they are fitted to 2.5 and 3 % rms)."""
    for kind, size, tiles, us in ((ops.ROWS_GATED, (2011, 12288, 2048), 13, 88.0), (ops.ROWS_GATED, (1500, 12288, 2048), 10, 72.8), (ops.ROWS_GATED, (409, 19456, 2560), 9, 43.0),
                                  (ops.ROWS_GATED, (2048, 24576, 4096), 16, 293.0), (ops.ROWS_STORE, (2048, 6144, 4096), 13, 75.5), (ops.ROWS_STORE, (1356, 8192, 4096), 11, 69.1),
                                  (ops.ROWS_STORE, (1356, 8192, 4096), 13, 79.0)):
        assert abs(ops._rows_tall_us(*size, tiles, 1, kind) / us - 1) < 0.1, (size, tiles)
    for size, tiles, us in (((2011, 12288, 2048), 8, 88.0), ((1500, 12288, 2048), 6, 76.0), ((1356, 12288, 2048), 6, 71.2), ((409, 19456, 2560), 5, 56.0), ((1356, 19456, 2560), 7, 119.7)):
        assert abs(ops._rows_gated_us(*size, tiles) / us - 1) < 0.1, size
    assert ops._rows_gated_us(640, 12288, 2048, 8) is None                       # (one block a unit)


def test_products_that_tall_blocks_made_slower_go_by_what_stood_there():
    gated = lambda M, N, K: ops.rows_product_tall(M, N, K, ops.ROWS_GATED, ops.rows_product_gated(M, N, K, True))
    stored = lambda M, N, K: ops.rows_product_tall(M, N, K, ops.ROWS_STORE, ops.rows_product_stored(M, N, K))
    # the rows of a second round that is part empty, against small blocks
    assert [gated(M, 12288, 2048) for M in (1500, 1700, 1790, 2011)] == [None] * 4 and gated(1356, 19456, 2560) is None and gated(1000, 24576, 4096) is None
    assert gated(1000, 8192, 2048) is None and gated(1200, 12288, 2048) == (15, 1) and gated(1356, 12288, 2048) == (9, 1)
    # one row tile fewer than 409 rows have
    assert gated(385, 19456, 2560) == gated(409, 19456, 2560) == (9, 1)
    # many rows: the library's tiles
    assert gated(8192, 24576, 4096) is None and [stored(M, 4096, 1024) for M in (3400, 4000, 8192, 16384)] == [None] * 4
    assert stored(8192, 4096, 2048) is None and stored(3600, 2048, 2048) is None and stored(4200, 2048, 6144) is None
    # stored small blocks, one a unit
    assert stored(1600, 4096, 1024) is None and stored(1600, 4096, 2048) is None and stored(800, 8192, 2048) is None
    # row tiles by what all units do, not by whether a round is full to the last block
    assert stored(1356, 8192, 4096) == (11, 1) and stored(1500, 8192, 2048) == (12, 1)
    assert ops.rows_product_tall(1500, 4096, 12288, ops.ROWS_PARTS) == (12, 2)
