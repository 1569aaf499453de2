"""Products of many rows whose columns' blocks are of two sizes (csrc/gemm_rows.hip): two blocks and more a compute unit, rows that are
dealt evenly and that are not, a last tile of rows that is part empty."""
import pytest
import torch

from tests.gpu_util import close, require_gpu

pytestmark = pytest.mark.gpu


# (M, N, K, row tiles): 2 blocks of 4 + 3 tiles, 3 of 5 + 4 + 4, 5 of 5 + 4 ..., 6 of 6 and 5, 4 of 8 and 7 tiles a column
@pytest.mark.parametrize("M,N,K,tiles", [(100, 33280, 128, 4), (200, 25632, 256, 5), (333, 23040, 128, 8), (545, 13312, 128, 6), (498, 33280, 128, 8)])
@pytest.mark.parametrize("how", ["stored", "gated", "parts"])
def test_blocks_of_two_sizes(M, N, K, tiles, how, monkeypatch):
    from spyinfer_amd.kernels import ops
    dev = require_gpu()
    g = torch.Generator().manual_seed(M + N)
    x, w = torch.randn((M, K), generator=g).bfloat16(), (torch.randn((N, K), generator=g) * K ** -0.5).bfloat16()
    xd, wd = x.to(dev), w.to(dev)
    tiled, want = ops.tile_weight(wd), xd.double() @ wd.double().t()
    if how == "stored":
        monkeypatch.setattr(ops, "rows_product_stored", lambda *size: tiles)
        close(ops.linear(xd, wd, tiled=tiled), want, torch.bfloat16, what="stored")
    elif how == "gated":
        monkeypatch.setattr(ops, "rows_product_gated", lambda *size: tiles)
        a, up = want[:, :N // 2], want[:, N // 2:]
        close(ops.linear_swiglu(xd, wd, tiled), torch.nn.functional.silu(a) * up, torch.bfloat16, what="gated")
    else:
        monkeypatch.setattr(ops, "rows_product_parts", lambda *size: (tiles, K // 128))
        out = ops.linear_parts(xd, wd, tiled)
        # (products of bfloat16 values summed in float32 over at most 256 of them)
        assert float((out.parts.double().sum(0) - want).abs().max()) < 1e-5 * 10
