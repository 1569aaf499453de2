"""Products that leave their results in parts, through the blocks and norms of a model: every reader of parts against the same step without
them, and against plain float32 arithmetic."""
import types

import pytest
import torch

from tests.gpu_util import close, require_gpu

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", ["bfloat16", "float32"])
def test_a_model_with_its_products_in_parts(dtype, tmp_path, monkeypatch):
    """o and down of two blocks in parts of uneven length, summed by the block's second norm, the next block's first and the final norm with
    picked rows; the same step with every product whole."""
    from spyinfer_amd.engine.batch import StepEntry
    from spyinfer_amd.engine.runner import ModelRunner, load_model
    from spyinfer_amd.kernels import ops
    from spyinfer_amd.weights import write_random_model
    from tests.configs import INIT, TINY_E
    dev = require_gpu()
    folder = write_random_model(str(tmp_path / "model"), TINY_E, seed=4, dtype=torch.bfloat16, **INIT)
    runner = ModelRunner(load_model(folder, dtype, dev), dtype, dev, 16, 32, 4)
    summed, real = [], ops.add_parts_rms_norm

    def spy(resid, addend, weight, eps, out_dtype, rows=None):
        summed.append((addend.parts.shape[0], rows is not None))
        return real(resid, addend, weight, eps, out_dtype, rows)
    monkeypatch.setattr(ops, "add_parts_rms_norm", spy)

    def logits(parts):
        monkeypatch.setattr(ops, "rows_product_parts", lambda M, N, K: (5, parts) if parts else None)
        monkeypatch.setattr(ops, "f32_product_parts", lambda M, N, K: parts)
        live = [runner.manager.admit(name) for name in ("a", "b")]
        for rc, n in zip(live, (90, 45)):
            runner.manager.reserve(rc, n)
        out = runner.step([StepEntry(live[0], [(7 * i) % 590 for i in range(90)], (3, 89)), StepEntry(live[1], [(11 * i) % 590 for i in range(45)], (44,))]).clone()
        for rc in live:
            runner.manager.release(rc)
        return out

    whole = logits(None)
    assert not summed
    in_parts = logits(3)
    assert summed == [(3, False)] * 3 + [(3, True)]
    # (both passes round their activations, each by itself: twice the bound of one)
    close(in_parts, whole, getattr(torch, dtype), scale=2.0, what="logits of a step with products in parts")


def addend(T, H, parts=3, seed=1):
    g = torch.Generator().manual_seed(seed)
    return torch.randn((T, H), generator=g), torch.randn((parts, T, H), generator=g)


def normed(x, w, eps, groups=1):
    xg = x.reshape(x.shape[0], groups, -1)
    return (xg / torch.sqrt((xg * xg).mean(-1, keepdim=True) + eps)).reshape(x.shape) * w


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("case", ["plain", "rows", "second", "groups", "odd", "off", "entry", "layer"])
def test_readers_of_parts(case, dtype):
    """A norm that sums parts in its pass, and the ways of those that do not: a second norm of the same sum, groups, a row that is no multiple
    of four, a weight off 16 bytes, what meets the stream at a walk's start, a layer norm."""
    from spyinfer_amd.kernels import ops
    from spyinfer_amd.parts import LayerNorm, RMSNorm
    dev = require_gpu()
    T, H = 67, 130 if case == "odd" else 256
    resid, y = addend(T, H)
    g = torch.Generator().manual_seed(5)
    weight = (1 + 0.1 * torch.randn((H,), generator=g)).to(dtype)
    w = weight.float()
    norm = LayerNorm(H, 1e-5) if case == "layer" else RMSNorm(H, 1e-5, groups=2 if case == "groups" else 1)
    off = torch.empty((H + 1,), dtype=dtype, device=dev)[1:]
    off.copy_(weight)
    norm.weight = off if case == "off" else weight.to(dev)
    parts, stream, total = ops.ProductParts(y.to(dev)), resid.to(dev), resid + y.sum(0)
    if case == "rows":
        rows = torch.tensor([66, 0, 9], dtype=torch.int32)
        close(norm.add_norm(stream, parts, dtype, rows.to(dev)), normed(total, w, 1e-5)[rows.long()], dtype, what="picked rows")
        assert torch.equal(stream.cpu(), resid)
        return
    if case == "second":
        other = RMSNorm(H, 1e-5)
        other.weight = (norm.weight.float() * 2.0).to(dtype)
        a, b = norm.add_norm(stream, parts, dtype, second=other)
        close(b, normed(total, 2.0 * w, 1e-5), dtype, scale=2.0, what="the second norm")
    elif case == "entry":
        base, vec = addend(T, H, 1, seed=9)
        total = total + base + vec[0, 0]
        a = norm.add_norm(stream, ops.EntryAddends(parts, base.to(dev), vec[0, 0].to(dev)), dtype)
    elif case == "layer":
        norm.bias = torch.zeros_like(norm.weight)
        a = norm.add_norm(stream, parts, dtype)
    else:
        a = norm.add_norm(stream, parts, dtype)
    # (rounded to the activations' type before the sum where the norm does not take parts, as a whole product is)
    close(stream, total, torch.float32 if case in ("plain", "layer") else dtype, what="the stream")
    ref = torch.nn.functional.layer_norm(total, (H,), w, None, 1e-5) if case == "layer" else normed(total, w, 1e-5, norm.groups)
    close(a, ref, dtype, scale=2.0, what="the norm")


def test_parts_before_a_block_that_adds_them_itself():
    """``OutputNormBlock`` after a block that left parts, alone and beside what meets the stream at a walk's start."""
    from spyinfer_amd.kernels import ops
    from spyinfer_amd.parts import OutputNormBlock, RMSNorm
    from spyinfer_amd.parts.base import Mixer
    dev = require_gpu()

    class Twice(Mixer):
        def forward(self, x, batch, cache, store=True):
            return 2.0 * x

    resid, y = addend(70, 128)
    norm = RMSNorm(128, 1e-5)
    norm.weight = torch.ones((128,), device=dev)
    base, vec = addend(70, 128, 1, seed=3)
    for entry in (False, True):
        pending = ops.ProductParts(y.to(dev))
        total = resid + y.sum(0)
        if entry:
            pending, total = ops.EntryAddends(pending, base.to(dev), vec[0, 0].to(dev)), total + base + vec[0, 0]
        batch = types.SimpleNamespace(act_dtype=torch.float32, shared={})
        out, left = OutputNormBlock(Twice(), norm).forward(resid.to(dev), pending, batch, None)
        assert left is None
        close(out, total + normed(2.0 * total, 1.0, 1e-5), torch.float32, what="the stream behind the block")
