"""The gated activation where its result is rounded to bfloat16 (csrc/common.h, gated_value_short) against 64 bits: every gate value of
bfloat16 from 2^-8 to 90, small gates beside exponentials close to overflow, in the activation pass, in products of many rows and of one
row tile.  A result has to be what a value within a few units of 2^-24 of the exact one rounds to."""
import pytest
import torch

from tests.gpu_util import require_gpu

pytestmark = pytest.mark.gpu


def gates(dev):
    z = torch.arange(0x3b80, 0x42b4, dtype=torch.int32).to(torch.int16).view(torch.bfloat16)             # 2^-8 .. 90
    return torch.cat([z, -z, torch.zeros(8, dtype=torch.bfloat16)]).to(dev)


def check(out, z, up, activation):
    """out [T, I] for gates z [T] and the other halves up [I]"""
    z, up, out = z.double()[:, None], up.double()[None], out.double()
    c1, c3 = (1.0, 0.0) if activation == "silu" else (1.5957691216057308, 0.07135481282553525)
    s = -z * (c1 + c3 * z * z)
    want = z / (1 + torch.exp(s)) * up
    # silu: the exponential, its sum with one, the quotient and the last product are within five units of 2^-24 altogether; the other one's exponent is
    # rounded three times before, c1 and c3 once each: 2.5 units of |s|.  One more for the rounding of the limits to float32 below
    units = 6.0 + (0.0 if activation == "silu" else 2.5) * s.abs()
    lo, hi = want - want.abs() * units * 2.0 ** -24, want + want.abs() * units * 2.0 ** -24
    lo, hi = lo.float().bfloat16().double(), hi.float().bfloat16().double()
    over = (s > 88.72).expand_as(want)                                         # the exponential overflows: the result is zero, below 1e-36
    ok = torch.where(over, (out.abs() <= torch.maximum(lo.abs(), hi.abs())), (lo <= out) & (out <= hi))
    # (numbers below bfloat16's normal ones: within the smallest of them)
    ok |= (out - want).abs() <= 2.0 ** -133
    bad = (~ok).nonzero()
    assert bad.shape[0] == 0, (bad.shape[0], float(z[bad[0, 0], 0]), float(up[0, bad[0, 1]]), float(out[tuple(bad[0])]), float(want[tuple(bad[0])]))


@pytest.mark.parametrize("activation", ["silu", "gelu_tanh"])
def test_activation_pass(activation):
    from spyinfer_amd.kernels import ops
    dev = require_gpu()
    z = gates(dev)
    up = torch.randn(256, generator=torch.Generator().manual_seed(1)).bfloat16().to(dev)
    out = ops.swiglu(torch.cat([z[:, None].expand(-1, 256), up[None].expand(z.shape[0], -1)], 1).contiguous(), activation)
    check(out, z, up, activation)


@pytest.mark.parametrize("activation", ["silu", "gelu_tanh"])
@pytest.mark.parametrize("rows", ["many", "16", "1"])
def test_products(rows, activation, monkeypatch):
    """Two of 128 numbers of a row are set: the gate's value, which the matrix passes on, and a one that it multiplies by the other half's."""
    from spyinfer_amd.kernels import ops
    dev = require_gpu()
    z = gates(dev)
    if rows != "many":
        z = z[(z < -80) | (z > 88)][:: 3 if rows == "16" else 15]
    up = torch.randn(256, generator=torch.Generator().manual_seed(2)).bfloat16().to(dev)
    x, w = torch.zeros((z.shape[0], 128), dtype=torch.bfloat16, device=dev), torch.zeros((512, 128), dtype=torch.bfloat16, device=dev)
    x[:, 5], x[:, 100], w[:256, 5], w[256:, 100] = z, 1.0, 1.0, up
    tiled = ops.tile_weight(w)
    monkeypatch.setattr(ops, "rows_product_gated", lambda *size: 8)
    step = z.shape[0] if rows == "many" else int(rows)
    out = torch.cat([ops.linear_swiglu(x[i:i + step].contiguous(), w, tiled, activation=activation) for i in range(0, z.shape[0], step)])
    check(out, z, up, activation)


@pytest.mark.parametrize("activation", ["silu", "gelu_tanh"])
def test_infinities_and_nan(activation):
    """As in float32, whose activation is the library's functions."""
    from spyinfer_amd.kernels import ops
    dev = require_gpu()
    z = torch.tensor([float("inf"), float("-inf"), float("nan"), 1e30, -1e30, 3e38, -3e38, -89.0, -1e4, 0.0, -0.0, 1e-38])
    up = torch.tensor([1.0, -2.0, float("inf"), float("nan"), 0.0, 1e-30, 3e38, 7.0])
    gate_up = torch.cat([z[:, None].expand(-1, 8), up[None].expand(12, -1)], 1).bfloat16().contiguous().to(dev)
    out, want = ops.swiglu(gate_up, activation), ops.swiglu(gate_up.float(), activation).bfloat16()
    assert torch.equal(out.isnan(), want.isnan()) and torch.equal(out[~want.isnan()], want[~want.isnan()])
