"""Per-head products whose K the waves of a block share (csrc/latent_attention.hip): K that ends inside a wave's part and before it, columns and
tokens that end inside a tile, several token tiles a block."""
import pytest
import torch

from tests.gpu_util import require_gpu

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("out_dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("T,H,N,K", [(1, 2, 17, 136), (5, 16, 128, 512), (16, 3, 16, 256), (33, 4, 31, 264), (130, 40, 33, 504), (64, 70, 128, 384)])
def test_products(T, H, N, K, out_dtype):
    from spyinfer_amd.kernels import ops
    dev = require_gpu()
    g = torch.Generator().manual_seed(T + H + N + K)
    x, w = torch.randn((T, H, K), generator=g).bfloat16(), (torch.randn((H, N, K), generator=g) / K ** 0.5).bfloat16()
    out = torch.full((T, H, N + 3), float("nan"), dtype=out_dtype, device=dev)
    ops.head_products(x.to(dev), H * K, K, w.to(dev), out, H * (N + 3), N + 3, T)
    a, b = x.double().transpose(0, 1), w.double().transpose(1, 2).contiguous()
    want, sizes = torch.bmm(a, b).transpose(0, 1), torch.bmm(a.abs(), b.abs()).transpose(0, 1)
    # K roundings of 24 bits at most, and one of the result's
    limit = (K + 8) * 2.0 ** -24 * sizes + (2.0 ** -8 * want.abs() if out_dtype == torch.bfloat16 else 0)
    got = out.double().cpu()
    assert bool(((got[:, :, :N] - want).abs() <= limit).all()) and bool(got[:, :, N:].isnan().all())
