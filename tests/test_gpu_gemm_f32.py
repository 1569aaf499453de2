"""The float32 products (csrc/gemm_f32.hip) at the edges of their kernels: numbers of rows around every tile, columns and K that are
multiples of nothing (K: of four), each choice of the dispatch."""
import pytest
import torch

from tests.gpu_util import close, require_gpu

pytestmark = pytest.mark.gpu

# (M, N, K): few rows with one, two and four rows of W a wave, whole and cut groups of K; row tiles one, two and four per block, several
# groups of them; tiles of 64 x 64 with K in four, two and one part
SHAPES = [(1, 1, 4), (1, 1023, 1028), (2, 12289, 260), (2, 20001, 512), (3, 7, 3076), (4, 2048, 2048), (4, 2049, 2304), (4, 12291, 516),
          (5, 1024, 1540), (8, 1000, 68), (8, 1025, 68), (9, 16, 64), (16, 33, 4), (17, 4100, 580), (31, 8200, 64), (33, 17, 1000), (50, 4097, 132),
          (64, 5000, 36), (65, 64, 2052), (129, 1030, 100), (64, 10177, 60), (65, 5121, 64), (700, 1023, 28), (130, 5440, 4), (129, 10890, 68), (1030, 2051, 96)]


@pytest.mark.parametrize("M,N,K", SHAPES)
def test_float32_product(M, N, K):
    from spyinfer_amd.kernels import ops
    dev = require_gpu()
    g = torch.Generator().manual_seed(M + 3 * N + 7 * K)
    x, w = torch.randn((M, K), generator=g).to(dev), torch.randn((N, K), generator=g).to(dev)
    held = torch.full((M * N + 4096,), float("nan"), device=dev)          # what lies behind the result stays as it is
    out = ops.linear(x, w, out=held[:M * N].view(M, N))
    # no product is rounded more often than a chain of 256 (or K / 8, the waves that share K) and the few sums of chains are:
    # |error| <= (roundings) 2^-24 sum |x w|
    bound = (max(256, K / 8) + K / 256 + 32) * 2.0 ** -24 * (x.double().abs() @ w.double().abs().t())
    assert bool(((out.double() - x.double() @ w.double().t()).abs() <= bound).all())
    assert bool(held[M * N:].isnan().all())


@pytest.mark.parametrize("M", [1, 30, 300])
def test_unaligned_operands_give_the_same_product(M):
    """Rows that do not begin at a multiple of 16 bytes are taken too (by the plain kernel)."""
    from spyinfer_amd.kernels import ops
    dev = require_gpu()
    g = torch.Generator().manual_seed(M)
    x, w = torch.randn((M, 64), generator=g).to(dev), torch.randn((1600, 64), generator=g).to(dev)
    odd = torch.empty(1600 * 64 + 1, device=dev)[1:].view(1600, 64)
    odd.copy_(w)
    bound = 2 * (256 + 32) * 2.0 ** -24 * (x.double().abs() @ w.double().abs().t())
    assert bool(((ops.linear(x, odd).double() - ops.linear(x, w).double()).abs() <= bound).all())


@pytest.mark.parametrize("M,N", [(1, 512), (40, 512), (300, 1100)])
def test_infinities_and_nan_stay_in_their_rows(M, N):
    from spyinfer_amd.kernels import ops
    dev = require_gpu()
    x, w = torch.ones((M, 100), device=dev), torch.ones((N, 100), device=dev)
    x[M - 1, 3], w[N - 1, 7], w[0, 99] = float("inf"), float("nan"), float("-inf")
    assert torch.equal(ops.linear(x, w).isnan(), (x @ w.t()).isnan())
    assert torch.equal(ops.linear(x, w).isinf(), (x @ w.t()).isinf())


@pytest.mark.parametrize("activation", ["silu", "gelu_tanh"])
@pytest.mark.parametrize("M,I,K", [(1, 5, 4), (1, 1023, 1028), (2, 130, 516), (3, 64, 2048), (4, 1001, 260), (4, 6144, 512)])
def test_gated_float32_product_of_few_rows(M, I, K, activation):
    from spyinfer_amd.kernels import ops
    dev = require_gpu()
    g = torch.Generator().manual_seed(M + I + K)
    x, w = torch.randn((M, K), generator=g), torch.randn((2 * I, K), generator=g) * K ** -0.5
    h = x.double() @ w.double().T
    act = torch.nn.functional.silu if activation == "silu" else lambda z: torch.nn.functional.gelu(z, approximate="tanh")
    close(ops.linear_swiglu(x.to(dev), w.to(dev), activation=activation), act(h[:, :I]) * h[:, I:], torch.float32, what="gated float32 product")
