"""Products of many rows by blocks of more than eight row tiles (csrc/gemm_rows_tall.hip): one turn of K, two, odd and even numbers of them, parts of
uneven length, every number of row tiles, a last tile of rows that reaches back, columns that are no multiple of a block's; against float64."""
import pytest
import torch

from tests.gpu_util import close, require_gpu

pytestmark = pytest.mark.gpu

SIZES = [(9, 144, 272, 128), (10, 317, 1040, 384), (11, 176, 48, 640), (12, 1300, 256, 256), (13, 409, 512, 1280), (14, 447, 768, 896), (15, 240, 256, 512), (16, 511, 528, 1152)]


def _operands(M, N, K):
    dev = require_gpu()
    g = torch.Generator().manual_seed(M + N)
    x, w = torch.randn((M, K), generator=g).bfloat16(), (torch.randn((N, K), generator=g) * K ** -0.5).bfloat16()
    wd = w.to(dev)
    return x, w, x.to(dev), wd


@pytest.mark.parametrize("tiles,M,N,K", SIZES)
def test_stored(tiles, M, N, K, monkeypatch):
    from spyinfer_amd.kernels import ops
    monkeypatch.setattr(ops, "rows_product_tall", lambda *size: (tiles, 1))
    x, w, xd, wd = _operands(M, N, K)
    close(ops.linear(xd, wd, tiled=ops.tile_weight(wd)), x.double() @ w.double().T, torch.bfloat16, what="product of many rows")


@pytest.mark.parametrize("tiles,M,N,K", SIZES)
def test_parts(tiles, M, N, K, monkeypatch):
    from spyinfer_amd.kernels import ops
    x, w, xd, wd = _operands(M, N, K)
    tiled = ops.tile_weight(wd)
    for parts in sorted({1, min(3, K // 128), K // 128}):
        monkeypatch.setattr(ops, "rows_product_tall", lambda *size: (tiles, parts))
        out = ops.linear_parts(xd, wd, tiled)
        assert isinstance(out, ops.ProductParts) and tuple(out.parts.shape) == (parts, M, N)
        # exact products of bfloat16 values, K float32 sums of terms of size K^-1/2: an error of some 2^-24 sqrt(K) terms' sizes
        bounds = [K // 128 * p // parts * 128 for p in range(parts + 1)]
        for p, (a, b) in enumerate(zip(bounds, bounds[1:])):
            ref = x[:, a:b].double() @ w[:, a:b].double().T
            assert float((out.parts[p].cpu().double() - ref).abs().max()) < 1e-5


@pytest.mark.parametrize("activation", ["silu", "gelu_tanh"])
@pytest.mark.parametrize("tiles,M,I,K", SIZES)
def test_gated(tiles, M, I, K, activation, monkeypatch):
    from spyinfer_amd.kernels import ops
    monkeypatch.setattr(ops, "rows_product_tall", lambda *size: (tiles, 1))
    x, w, xd, wd = _operands(M, 2 * I, K)
    out = ops.linear_swiglu(xd, wd, ops.tile_weight(wd), activation=activation)
    h = x.double() @ w.double().T
    act = torch.nn.functional.silu if activation == "silu" else lambda z: torch.nn.functional.gelu(z, approximate="tanh")
    close(out, act(h[:, :I]) * h[:, I:], torch.bfloat16, what="gated product of many rows")


def test_not_a_number_stays_in_its_row():
    """Rows that a block's last tile shares with the one before, and rows beside a NaN and an infinity."""
    from spyinfer_amd.kernels import ops
    x, w, xd, wd = _operands(1500, 6144, 2560)
    assert ops.rows_product_tall(1500, 6144, 2560, ops.ROWS_STORE) is not None
    xd[700, 3], xd[1499, 2559] = float("nan"), float("inf")
    out = ops.linear(xd, wd, tiled=ops.tile_weight(wd))
    bad = ~torch.isfinite(out).all(dim=1)
    assert bad.nonzero()[:, 0].tolist() == [700, 1499]
    keep = torch.ones(1500, dtype=torch.bool)
    keep[[700, 1499]] = False
    close(out[keep.to(out.device)], x[keep].double() @ w.double().T, torch.bfloat16, what="rows beside")
