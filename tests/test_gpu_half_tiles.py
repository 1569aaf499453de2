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
