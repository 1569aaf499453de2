"""Results of products that still lie in parts, on their way from a block to the norm that sums them."""
import pytest
import torch

from spyinfer_amd.parts import LayerNorm, RMSNorm


@pytest.mark.parametrize("size,groups,offset,takes", [(128, 1, 0, True), (8192, 1, 0, True), (516, 1, 4, True), (128, 2, 0, False), (130, 1, 0, False),
                                                      (8196, 1, 0, False), (128, 1, 1, False)])
def test_a_norm_that_cannot_sum_parts_does_not_ask_for_them(size, groups, offset, takes):
    norm = RMSNorm(size, 1e-6, groups=groups)
    assert not norm.takes_product_parts                              # (no weight yet)
    norm.weight = torch.ones(size + offset)[offset:]
    assert norm.takes_product_parts == takes


def test_a_norm_with_a_sum_of_its_own_gets_none():
    class Own(RMSNorm):
        def add_norm(self, resid, delta, out_dtype, rows=None):
            return super().add_norm(resid, delta, out_dtype, rows)

    norm = Own(128, 1e-6)
    norm.weight = torch.ones(128)
    assert not norm.takes_product_parts and not getattr(LayerNorm(128, 1e-6), "takes_product_parts", False)


def test_parts_are_added_like_a_tensor():
    """What a block of another arrangement may do with an addend that is pending."""
    from spyinfer_amd.kernels import ops
    y = torch.randn((3, 5, 8), generator=torch.Generator().manual_seed(2))
    parts, stream, total = ops.ProductParts(y), torch.randn((5, 8)), y.sum(0)
    assert tuple(parts.shape) == (5, 8) and parts.dtype == torch.float32 and parts.device == y.device
    for out in (stream + parts, parts + stream, torch.add(stream, parts), stream.clone().add_(parts), stream.clone().add_(parts.float()),
                stream + parts.to(torch.float32)):
        assert torch.equal(out, stream + total)
    held = stream.clone()
    held += parts
    assert torch.equal(held, stream + total)
    assert torch.equal(torch.cat([parts.to(torch.float64), total.double()]), torch.cat([total.double(), total.double()]))
