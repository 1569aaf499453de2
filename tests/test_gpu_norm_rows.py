"""Norms that sum addends (csrc/elementwise.hip): rows of one piece a thread and of several, on both sides of the line by the number of
values, a last wave that is part empty; addends in parts, fewer and more than a thread asks for at once."""
import pytest
import torch

from tests.gpu_util import require_gpu

pytestmark = pytest.mark.gpu


def limit(want, dtype, H):
    # a tree of H squares and a handful of roundings; a bfloat16 result is rounded once
    return (2.0 ** -24 * (H ** 0.5 + 16) + (2.0 ** -8 if dtype == torch.bfloat16 else 0.0)) * want.abs() + 1e-30


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("T,H", [(1, 4), (3, 252), (5, 1028), (2, 4096), (3, 4100), (2, 8192), (2, 8196), (2, 16388), (600, 4096), (1030, 2048)])
def test_add_rms_norm(T, H, dtype):
    from spyinfer_amd.kernels import ops
    dev = require_gpu()
    g = torch.Generator().manual_seed(T + H)
    x, y, w = torch.randn((T, H), generator=g), torch.randn((T, H), generator=g).to(dtype), torch.randn((H,), generator=g).to(dtype)
    resid = x.to(dev)
    out = ops.add_rms_norm(resid, y.to(dev), w.to(dev), 1e-5, dtype)
    s = x + y.float()
    assert torch.equal(resid.cpu(), s)
    want = s.double() * torch.rsqrt(s.double().pow(2).mean(1, keepdim=True) + 1e-5) * w.double()
    assert bool(((out.cpu().double() - want).abs() <= limit(want, dtype, H)).all())


@pytest.mark.parametrize("parts", [1, 2, 3, 4, 6, 7, 12])
@pytest.mark.parametrize("T,H", [(2, 4), (3, 1028), (2, 4096), (2, 4100), (2, 8192)])
def test_parts(T, H, parts):
    from spyinfer_amd.kernels import ops
    dev = require_gpu()
    g = torch.Generator().manual_seed(T + H + parts)
    x, y, w = torch.randn((T, H), generator=g), torch.randn((parts, T, H), generator=g), torch.randn((H,), generator=g)
    resid = x.to(dev)
    out = ops.add_parts_rms_norm(resid, ops.ProductParts(y.to(dev)), w.to(dev), 1e-5, torch.float32)
    s = y[0]
    for p in range(1, parts):
        s = s + y[p]                                    # in the order of the parts, the stream last
    s = x + s
    assert torch.equal(resid.cpu(), s)
    want = s.double() * torch.rsqrt(s.double().pow(2).mean(1, keepdim=True) + 1e-5) * w.double()
    assert bool(((out.cpu().double() - want).abs() <= limit(want, torch.float32, H)).all())


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("H", [252, 512, 700, 1028, 2048, 2560, 4096, 4100, 5120, 8192, 8196, 16388])
def test_a_row_is_the_same_bits_in_steps_of_every_size(H, dtype):
    from spyinfer_amd.kernels import ops
    dev = require_gpu()
    T, few = (2 << 20) // H + 1, 3
    g = torch.Generator().manual_seed(H)
    x, y, w = (torch.randn(s, generator=g) for s in ((T, H), (T, H), (H,)))
    x, y, w = x.to(dev), y.to(dtype).to(dev), w.to(dtype).to(dev)
    streams, outs = [], []
    for t in (T, few):
        streams.append(x[:t].clone())
        outs.append(ops.add_rms_norm(streams[-1], y[:t].clone(), w, 1e-5, dtype))
    assert torch.equal(streams[0][:few], streams[1]) and torch.equal(outs[0][:few], outs[1])
