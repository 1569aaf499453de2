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
