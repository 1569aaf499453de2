"""Float32 products of up to 32 rows that a block keeps in registers (csrc/gemm_f32.hip) against 64 bits: both numbers of row tiles, every length
of K a wave holds, tiles of W that end inside, blocks with one tile more than others, parts of K."""
import pytest
import torch

from tests.gpu_util import require_gpu

pytestmark = pytest.mark.gpu


def bound(x, w, parts=1):
    # a wave's chain is K / 8 of a part long, eight waves and the parts follow
    return (x.shape[1] / 8 / parts + 8 + parts) * 2.0 ** -24 * (x.double().abs() @ w.double().abs().t())


def operands(M, N, K):
    dev, g = require_gpu(), torch.Generator().manual_seed(M + 3 * N + 7 * K)
    return torch.randn((M, K), generator=g).to(dev), (torch.randn((N, K), generator=g) * K ** -0.5).to(dev)


@pytest.mark.parametrize("M", [5, 8, 9, 16, 17, 32])
@pytest.mark.parametrize("N,K", [(4097, 512), (4112, 1024), (8201, 1536), (4100, 2048), (12290, 1024)])
def test_product(M, N, K):
    from spyinfer_amd.kernels import ops
    x, w = operands(M, N, K)
    held = torch.full((M * N + 64,), float("nan"), device=x.device)
    out = ops.linear(x, w, out=held[:M * N].view(M, N))
    assert bool(((out.double() - x.double() @ w.double().t()).abs() <= bound(x, w)).all()) and bool(held[M * N:].isnan().all())


@pytest.mark.parametrize("activation", ["silu", "gelu_tanh"])
@pytest.mark.parametrize("M", [9, 16, 17, 32])
@pytest.mark.parametrize("I,K", [(2049, 512), (3000, 1024), (2055, 1536), (6144, 2048)])
def test_gated(M, I, K, activation):
    from spyinfer_amd.kernels import ops
    x, w = operands(M, 2 * I, K)
    h, err = x.double() @ w.double().t(), bound(x, w)
    act = torch.nn.functional.silu if activation == "silu" else lambda z: torch.nn.functional.gelu(z, approximate="tanh")
    a, up = act(h[:, :I]), h[:, I:]
    limit = 1.13 * err[:, :I] * (up.abs() + err[:, I:]) + a.abs() * err[:, I:] + 16 * 2.0 ** -24 * (h[:, :I] * up).abs() + 1e-30
    assert bool(((ops.linear_swiglu(x, w, activation=activation).double() - a * up).abs() <= limit).all())


@pytest.mark.parametrize("M", [9, 16, 17, 32])
@pytest.mark.parametrize("N,K,parts", [(1, 1024, 2), (17, 4608, 9), (1023, 2048, 4), (1024, 3072, 2), (2048, 6144, 12), (2050, 6144, 4), (4095, 4096, 2)])
def test_parts_of_k(M, N, K, parts):
    from spyinfer_amd.kernels import ops
    x, w = operands(M, N, K)
    assert ops.f32_rows_held(M, K, parts)
    held = torch.full((parts * M * N + 64,), float("nan"), device=x.device)
    ops.hip().call("spy_gemm_f32_parts", ops._ptr(held), ops._ptr(x), ops._ptr(w), M, N, K, parts, ops._Hip.stream())
    out = held[:parts * M * N].view(parts, M, N).double().sum(0)
    assert bool(((out - x.double() @ w.double().t()).abs() <= bound(x, w, parts)).all()) and bool(held[parts * M * N:].isnan().all())
    y = ops.linear_parts(x, w)
    if ops.f32_held_parts(M, N, K):
        assert y.parts.shape[0] == ops.f32_held_parts(M, N, K)
        assert bool(((y.parts.double().sum(0) - x.double() @ w.double().t()).abs() <= bound(x, w)).all())


@pytest.mark.parametrize("M", [9, 32])
def test_infinities_and_nan_stay_in_their_rows(M):
    from spyinfer_amd.kernels import ops
    dev = require_gpu()
    x, w = torch.ones((M, 1024), device=dev), torch.ones((4500, 1024), device=dev)
    x[M - 1, 1023], w[4499, 7], w[3, 1022], w[1030] = float("inf"), float("nan"), float("-inf"), 0.0
    want = x @ w.t()
    out = ops.linear(x, w)
    assert torch.equal(out.isnan(), want.isnan()) and torch.equal(out[~want.isnan()], want[~want.isnan()])
