"""Decode products of narrow matrices by blocks of half a column tile (csrc/gemm_decode.hip): few columns, chunks of K that fill a
wave's rounds and that do not, both hand-overs."""
import pytest
import torch

from tests.gpu_util import close, require_gpu

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M", [1, 5, 16])
@pytest.mark.parametrize("N,K", [(16, 128), (32, 1024), (1024, 2944), (1024, 3072), (2048, 3200), (2016, 6144)])
def test_half_tiles(M, N, K):
    from spyinfer_amd.kernels import ops
    dev = require_gpu()
    g = torch.Generator().manual_seed(M + N + K)
    x, w = torch.randn((M, K), generator=g).bfloat16(), (torch.randn((N, K), generator=g) * K ** -0.5).bfloat16()
    h, wn = torch.randn((M, N), generator=g), torch.randn((N,), generator=g).bfloat16()
    tiled, want = ops.tile_weight(w.to(dev)), x.double() @ w.double().t()
    close(ops.decode_linear(x.to(dev), tiled), want, torch.bfloat16, what="stored product")
    assert ops.residual_parts(M, N) == N // 8
    resid = h.to(dev)
    out = ops.decode_linear_residual(x.to(dev), tiled, resid, wn.to(dev), 1e-6)
    close(resid, h.double() + want, torch.float32, scale=4.0, what="stream")
    rows = out.xw.to_rows() if isinstance(out.xw, ops.OperandRows) else out.xw
    assert torch.equal(rows, (resid * wn.to(dev).float()).bfloat16())
    assert torch.allclose(out.ss_parts.sum(0)[:M], (resid * resid).sum(1), rtol=1e-5) and float(out.ss_parts[:, M:].abs().max() if M < 16 else 0.0) == 0.0


@pytest.mark.parametrize("M", [1, 3, 4, 8, 9, 16])
@pytest.mark.parametrize("K", [1024, 1152, 2048, 2176, 3200])
def test_both_sides_of_the_lines(M, K):
    """Whole tiles and halves: the same products, and parts of the sums of squares that add up, for rows as they lie and in operand order."""
    from spyinfer_amd.kernels import ops
    dev, N = require_gpu(), 1040
    g = torch.Generator().manual_seed(M + K)
    w, order = (torch.randn((N, K), generator=g) * K ** -0.5).bfloat16().to(dev), ops.OperandRows.empty(M, K, dev)
    order.data.copy_(torch.randn(order.data.shape, generator=g))
    x = order.to_rows()
    tiled, want = ops.tile_weight(w), x.double() @ w.double().t()
    close(ops.decode_linear(x, tiled), want, torch.bfloat16, what="rows")
    close(ops.decode_linear(order, tiled), want, torch.bfloat16, what="operand order")
    resid, wn = torch.randn((M, N), generator=g).to(dev), torch.ones(N, dtype=torch.bfloat16, device=dev)
    before = resid.double()
    out = ops.decode_linear_residual(order, tiled, resid, wn, 1e-6)
    assert out.ss_parts.shape[0] == (N // 16 if K == 1024 or (K == 2048 and M <= 8) else N // 8)
    close(resid, before + want, torch.float32, scale=4.0, what="stream")
    assert torch.allclose(out.ss_parts.sum(0)[:M], (resid * resid).sum(1), rtol=1e-5)
