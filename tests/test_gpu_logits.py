"""Logits of 9 to 208 bfloat16 rows: the kernels that walk column tiles (plain rows) and those of many rows, with float32 results."""
import pytest
import torch

from spyinfer_amd.kernels import ops

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


# the ends of the row tiles and of the rule's ranges; column tiles that fill no whole group, block or run; few and many a compute unit
@pytest.mark.parametrize("rows", [9, 10, 11, 16, 17, 18, 19, 32, 33, 48, 49, 63, 64, 65, 79, 80, 95, 127, 128, 129, 207, 208, 209])
@pytest.mark.parametrize("N,K", [(8208, 128), (32784, 384), (65552, 256), (73760, 1152)])
def test_logits(rows, N, K):
    gen = torch.Generator(device=DEV).manual_seed(rows + N)
    x = torch.randn((rows, K), generator=gen, device=DEV).bfloat16()
    w = torch.randn((N, K), generator=gen, device=DEV).bfloat16()
    out = torch.full((rows + 1, N), -5.0, device=DEV)
    ops.linear_few(x, w, ops.tile_weight(w), torch.float32, out[:rows])
    xd, wd = x.double(), w.double()
    # products of bfloat16 are exact in float32; K of them are added in some order: K roundings of 2^-24 of the sum of sizes at most
    assert bool(((out[:rows].double() - xd @ wd.t()).abs() <= K * 2.0 ** -24 * (xd.abs() @ wd.abs().t())).all())
    assert bool((out[rows] == -5.0).all())


def test_which_rows():
    assert [ops.rows_product_logits(m, 151936, 2560) for m in (63, 64, 79, 80, 128, 208, 209)] == [0, 4, 4, 5, 8, 8, 0]
    assert [ops.rows_product_logits(64, n, 2048) for n in (65520, 65536)] == [0, 4] and [ops.rows_product_logits(65, n, 2048) for n in (32752, 32768)] == [0, 4]
    assert ops.rows_product_logits(100, 65544, 2048) == 0 and ops.rows_product_logits(100, 65536, 2080) == 0 and ops.rows_product_logits(100, 262144, 4096) == 0


def test_blocks_of_a_column():
    # 128 columns of blocks: two blocks each find a unit; 129 and more: one block up to 128 rows
    assert [ops.rows_product_logits(m, 32768, 1024) for m in (80, 96, 127, 128, 160, 208)] == [4, 4, 4, 4, 5, 7]
    assert [ops.rows_product_logits(m, 33024, 1024) for m in (80, 96, 128)] == [5, 6, 8]
    # 784 blocks are three rounds and sixteen
    assert [ops.rows_product_logits(m, 100352, 2048) for m in (128, 129, 208)] == [8, 0, 0] and ops.rows_product_logits(129, 151936, 2048) == 8


@pytest.mark.parametrize("rows", [80, 96, 112, 128, 160])
def test_logits_of_two_blocks_a_column(rows):
    gen = torch.Generator(device=DEV).manual_seed(rows)
    x, w = torch.randn((rows, 384), generator=gen, device=DEV).bfloat16(), torch.randn((32768, 384), generator=gen, device=DEV).bfloat16()
    out = ops.linear_few(x, w, ops.tile_weight(w), torch.float32).double()
    xd, wd = x.double(), w.double()
    assert bool(((out - xd @ wd.t()).abs() <= 384 * 2.0 ** -24 * (xd.abs() @ wd.abs().t())).all())
