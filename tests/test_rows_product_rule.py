"""The sizes that go to the products of many rows, and what they are launched with: within what the kernel takes, for every size."""
import random
import threading

from spyinfer_amd.kernels import ops


def test_launches_fit_the_kernel():
    rng = random.Random(3)
    for _ in range(3000):
        M, N, K = int(2 ** rng.uniform(0, 14)), 16 * rng.randint(1, 2000), 128 * rng.randint(1, 120)
        plan = ops.rows_product_parts.__wrapped__(M, N, K)
        if plan is not None:
            tiles, parts = plan
            assert M > 64 and 4 <= tiles <= 8 and 16 * tiles <= M and 1 <= parts <= K // 256 and parts * M * N * 4 <= ops.PARTS_MAX_BYTES
            assert N * K < 1 << 30 and M * K < 1 << 30
        tiles = ops.rows_product_gated.__wrapped__(M, 2 * N, K, True)
        assert tiles == 0 or (M > 64 and 4 <= tiles <= 8 and 16 * tiles <= M and 2 * N * K < 1 << 30 and M * K < 1 << 30)
        tiles = ops.rows_product_stored.__wrapped__(M, N, K)
        assert tiles == 0 or (M > 64 and 4 <= tiles <= 8 and 16 * tiles <= M)
        parts = ops.f32_product_parts.__wrapped__(M, N, K)
        assert parts is None or (M > 16 and 2 <= parts <= K // 128 and parts * M * N * 4 <= ops.PARTS_MAX_BYTES)


def test_sizes_on_both_sides_of_the_line():
    assert ops.rows_product_parts(409, 2560, 9728) == (7, 6)
    assert ops.rows_product_parts(2011, 2560, 9728) is not None and ops.rows_product_parts(2011, 4096, 12288) is None
    assert ops.rows_product_parts(64, 2560, 9728) is None and ops.rows_product_parts(409, 2048, 2048) is None
    assert ops.rows_product_parts(200, 1024, 2048) is not None and ops.rows_product_parts(200, 1024, 1920) is None
    assert ops.rows_product_gated(1356, 12288, 2048, True) == 6 and ops.rows_product_gated(64, 12288, 2048, True) == 0
    assert ops.rows_product_gated(2011, 24576, 4096, True) == 0 and ops.rows_product_gated(2011, 24576, 4096, False) > 0
    assert ops.rows_product_gated(200, 6144, 4096, True) == 0
    assert ops.f32_product_parts(611, 1024, 2048) == 3 and ops.f32_product_parts(16, 1024, 2048) is None and ops.f32_product_parts(1500, 2048, 2048) is None
    assert ops.rows_product_stored(409, 4096, 1024) > 0 and ops.rows_product_stored(409, 4096, 2048) == 0 and ops.rows_product_stored(1356, 4096, 2048) > 0 and ops.rows_product_stored(1356, 6144, 1024) == 0


def test_replayed_steps_leave_the_host_s_time_out():
    for size in ((130, 4096, 1024), (409, 6144, 512), (640, 4096, 2048)):
        assert ops.rows_product_stored(*size) > 0 and ops.rows_product_stored(*size, True) == 0


def test_a_replayed_step_is_one_thread_s():
    seen = []
    with ops.replayed_step():
        with ops.replayed_step():
            pass
        other = threading.Thread(target=lambda: seen.append(ops._step.replayed))
        other.start()
        other.join()
        seen.append(ops._step.replayed)
    try:
        with ops.replayed_step():
            raise KeyError
    except KeyError:
        seen.append(ops._step.replayed)
    assert seen == [False, True, False]


def test_gated_products_go_to_the_side_that_was_measured_faster():
    slower = [(180, 9728, 2560), (409, 6144, 4096), (760, 4096, 4096), (240, 8192, 3072), (450, 6144, 5120), (288, 24576, 4096), (320, 24576, 4096),
              (450, 17408, 5120), (369, 27648, 5120), (561, 16384, 3072)]
    faster = [(409, 6144, 1024), (240, 9728, 2560), (500, 6144, 2560), (409, 19456, 2560), (1356, 12288, 2048), (561, 6144, 5120), (129, 17408, 5120),
              (450, 8192, 3072), (240, 24576, 4096), (561, 24576, 4096), (409, 27648, 5120), (640, 17408, 5120), (760, 6144, 4096)]
    assert [ops.rows_product_gated(*size, True) > 0 for size in slower] == [False] * len(slower)
    assert [ops.rows_product_gated(*size, True) > 0 for size in faster] == [True] * len(faster)
    assert all(ops.rows_product_gated(*size, False) > 0 for size in slower + faster)


def test_float32_products_in_parts_that_split_values():
    rng = random.Random(5)
    for _ in range(2000):
        M, N, K = int(2 ** rng.uniform(0, 12)), 4 * rng.randint(1, 4000), 32 * rng.randint(1, 400)
        parts = ops.f32_product_parts.__wrapped__(M, N, K)
        assert parts is None or (2 <= parts <= K // 128 and parts * M * N * 4 <= ops.PARTS_MAX_BYTES)
    assert ops.f32_rows_split(33, 8192, 1024) and not ops.f32_rows_split(32, 8192, 1024) and not ops.f32_rows_split(90, 4032, 1024)
    assert ops.f32_rows_split(90, 1024, 1024, 2) and not ops.f32_rows_split(600, 8192, 1000)
    assert ops.f32_product_parts(611, 1024, 3072) == 6 and ops.f32_product_parts(90, 2048, 2048) == 4
    # (long prompts too: more parts than small tiles would need)
    assert all(-(-M // 64) * (N // 64) * ops.f32_product_parts(M, N, K) > 1400 for M, N, K in ((1354, 2048, 6144), (802, 2560, 4096), (4096, 1024, 3072)))


def test_float32_products_in_parts_of_rows_that_are_held():
    rng = random.Random(6)
    for _ in range(2000):
        M, N, K = rng.randint(1, 40), rng.randint(1, 5000), rng.choice((1, 8, 64)) * 64 * rng.randint(1, 40)
        parts = ops.f32_held_parts.__wrapped__(M, N, K)
        assert parts is None or (8 < M <= 32 and N <= 4096 and 2 <= parts <= 12 and K % (512 * parts) == 0 and K // parts <= 2048)
    assert ops.f32_held_parts(16, 1024, 3072) == 6 and ops.f32_held_parts(16, 1024, 3000) is None and ops.f32_held_parts(33, 1024, 3072) is None
