"""When the experts' products go by groups of rows of one expert, and when a tile of 16 rows at a time: both sides of the line as
measured (microseconds a tile at a time / by groups in the comments), at the sizes where it is clear."""
import pytest


@pytest.mark.parametrize("pairs,experts,K,F,gated,groups", [
    (8, 1, 1024, 1024, True, False),            # 15 / 33: few blocks walk all of K
    (96, 1, 1024, 1024, True, False),           # 19 / 38
    (64, 8, 256, 512, True, False),             # 14 / 22
    (64, 2, 2048, 1536, True, False),           # 26 / 51
    (384, 8, 2048, 1536, True, True),           # 99 / 58
    (256, 8, 2048, 4096, True, True),           # 185 / 112
    (512, 32, 2048, 1536, True, True),          # 181 / 139
    (256, 32, 4096, 3072, True, True),          # 479 / 429
    (48, 32, 4096, 3072, True, False),          # (decoding: most experts have one tile)
    (128, 32, 2048, 1536, True, False),         # 127 / 137
    (1024, 64, 2048, 768, False, True),
    (8044, 32, 2048, 1536, True, True),
    (1 << 21, 1, 64, 64, True, True),           # (a tile at a time would be more blocks than a grid has)
    (15 * 12, 12, 720, 480, True, False),       # K and F no multiple of 64: from 16 rows an expert on
    (16 * 12, 12, 720, 480, True, True)])
def test_rule(pairs, experts, K, F, gated, groups):
    from spyinfer_amd.kernels import ops
    assert ops.experts_by_groups(pairs, experts, K, F, gated) is groups
