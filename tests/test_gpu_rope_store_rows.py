"""Per-head norm, rotation and store of many tokens (csrc/elementwise.hip's kernel with wide accesses) against the kernel of few tokens:
both types, every head size, pages filled in order, from the middle and out of order."""
import pytest
import torch

from tests.gpu_util import require_gpu

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("d,n_q,n_kv,T,normed", [(16, 3, 1, 64, True), (32, 4, 2, 77, False), (64, 6, 2, 130, True), (128, 5, 5, 211, True), (256, 2, 1, 65, False), (256, 2, 1, 260, True)])
@pytest.mark.parametrize("order", ["straight", "shifted", "mixed"])
def test_many_tokens(d, n_q, n_kv, T, normed, order, dtype):
    from spyinfer_amd.kernels import ops
    dev = require_gpu()
    P = 16
    g = torch.Generator().manual_seed(d + T)
    x = torch.randn((T, (n_q + 2 * n_kv) * d), generator=g).to(dev, dtype)
    qw, kw = [(1 + 0.1 * torch.randn((d,), generator=g)).to(dev, dtype) if normed else None for _ in range(2)]
    cos, sin = torch.randn((400, d // 2), generator=g).to(dev), torch.randn((400, d // 2), generator=g).to(dev)
    pages = T // P + 3
    slots = torch.arange(T) + (5 if order == "shifted" else 0)
    if order == "mixed":
        slots = torch.randperm(pages * P, generator=g)[:T]
        slots[3] = -1
    slots, pos = slots.int().to(dev), torch.arange(T).int().to(dev)

    def run(pieces):
        k, v = torch.zeros((pages, n_kv, P, d), device=dev, dtype=dtype), torch.zeros((pages, n_kv, d, P), device=dev, dtype=dtype)
        q = [ops.qk_norm_rope_store(x[a:b].contiguous(), n_q, n_kv, d, qw, kw, 1e-6, cos, sin, d, pos[a:b].contiguous(), k, v, P, slots[a:b].contiguous())
             for a, b in pieces]
        return torch.cat(q), k, v

    many, few = run([(0, T)]), run([(i, min(T, i + 40)) for i in range(0, T, 40)])
    for a, b in zip(many, few):
        # (sums of up to 256 squares in another order, then three roundings: 2^-18 of a value and its pair; in bfloat16 a rounding may fall the other way)
        tol = 2.0 ** -18 if dtype == torch.float32 else 2.0 ** -7
        assert bool(((a.float() - b.float()).abs() <= tol * (b.float().abs() + float(b.float().pow(2).mean().sqrt()))).all())
    assert torch.equal(many[2], few[2])                                            # values are only moved


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("order", ["straight", "mixed"])
def test_values_keep_their_bits(dtype, order):
    """Every number of bfloat16, NaN with all their bits among them, and as many of float32."""
    from spyinfer_amd.kernels import ops
    dev, T, d, P = require_gpu(), 512, 128, 16
    bits = torch.arange(65536, dtype=torch.int32)
    values = (bits << 16 | bits).view(torch.float32) if dtype == torch.float32 else bits.to(torch.int16).view(torch.bfloat16)
    x = torch.zeros((T, 3 * d), dtype=dtype)
    raw = torch.int32 if dtype == torch.float32 else torch.int16
    x.view(raw)[:, 2 * d:] = values.view(raw).view(T, d)
    slots = (torch.arange(T) if order == "straight" else torch.randperm(T, generator=torch.Generator().manual_seed(1))).int()
    k, v = torch.zeros((T // P, 1, P, d), device=dev, dtype=dtype), torch.zeros((T // P, 1, d, P), device=dev, dtype=dtype)
    table = torch.ones((T, d // 2), device=dev)
    ops.qk_norm_rope_store(x.to(dev), 1, 1, d, None, None, 1e-6, table, table, d, torch.arange(T, device=dev).int(), k, v, P, slots.to(dev))
    kept = v.view(raw).cpu().permute(0, 3, 1, 2).reshape(T, d)[slots.long()]
    assert torch.equal(kept, x.view(raw)[:, 2 * d:])
