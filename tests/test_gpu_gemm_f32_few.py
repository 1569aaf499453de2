"""Float32 products of up to eight rows (csrc/gemm_f32.hip) against 64 bits: every choice of rows of W and waves a block, columns that end
inside a block, K that ends inside a chunk, a wave's turn and a round."""
import pytest
import torch

from tests.gpu_util import require_gpu

pytestmark = pytest.mark.gpu

# (N, K): rows of W up to 1024, up to 4096, up to 8192, beyond; K of one chunk and less, chunks for some of the waves, whole rounds and a rest
SIZES = [(1, 4), (7, 256), (1023, 1300), (1024, 3072), (1027, 2048), (4093, 520), (4097, 2308), (8191, 768), (8200, 1028), (12290, 2052)]


def bound(x, w):
    # a lane's chain has K / 64 roundings at most, 64 lanes and eight waves are summed in a tree and a chain of 32
    return (x.shape[1] / 64 + 64) * 2.0 ** -24 * (x.double().abs() @ w.double().abs().t())


@pytest.mark.parametrize("M", [1, 2, 3, 4, 5, 8])
@pytest.mark.parametrize("N,K", SIZES)
def test_product(M, N, K):
    from spyinfer_amd.kernels import ops
    dev = require_gpu()
    g = torch.Generator().manual_seed(M + 3 * N + 7 * K)
    x, w = torch.randn((M, K), generator=g).to(dev), torch.randn((N, K), generator=g).to(dev)
    held = torch.full((M * N + 64,), float("nan"), device=dev)
    out = ops.linear(x, w, out=held[:M * N].view(M, N))
    # (5 to 8 rows, 4096 columns and more, K up to 1024 are the narrow kernel's: one chain a wave)
    limit = bound(x, w) * (4 if M > 4 and N >= 4096 and K <= 1024 else 1)
    assert bool(((out.double() - x.double() @ w.double().t()).abs() <= limit).all()) and bool(held[M * N:].isnan().all())


@pytest.mark.parametrize("N,K", [(1023, 2048), (1023, 4096), (1024, 4096), (1025, 4096), (300, 6144), (2048, 2052)])
def test_one_row(N, K):
    """Blocks of one row of W, one and two chunks a round, up to 4 million numbers of W, and one size beyond."""
    from spyinfer_amd.kernels import ops
    dev = require_gpu()
    g = torch.Generator().manual_seed(N + K)
    x, w = torch.randn((1, K), generator=g).to(dev), torch.randn((N, K), generator=g).to(dev)
    held = torch.full((N + 64,), float("nan"), device=dev)
    out = ops.linear(x, w, out=held[:N].view(1, N))
    assert bool(((out.double() - x.double() @ w.double().t()).abs() <= bound(x, w)).all()) and bool(held[N:].isnan().all())


@pytest.mark.parametrize("activation", ["silu", "gelu_tanh"])
@pytest.mark.parametrize("M", [1, 2, 4, 5, 7, 8])
@pytest.mark.parametrize("I,K", [(1, 4), (511, 1028), (2045, 512), (3072, 1024), (4101, 2048)])
def test_gated(M, I, K, activation):
    from spyinfer_amd.kernels import ops
    dev = require_gpu()
    g = torch.Generator().manual_seed(M + I + K)
    x, w = torch.randn((M, K), generator=g).to(dev), (torch.randn((2 * I, K), generator=g) * K ** -0.5).to(dev)
    h, err = x.double() @ w.double().t(), bound(x, w)
    act = torch.nn.functional.silu if activation == "silu" else lambda z: torch.nn.functional.gelu(z, approximate="tanh")
    a, up = act(h[:, :I]), h[:, I:]
    limit = 1.13 * err[:, :I] * (up.abs() + err[:, I:]) + a.abs() * err[:, I:] + 16 * 2.0 ** -24 * (h[:, :I] * up).abs() + 1e-30
    assert bool(((ops.linear_swiglu(x, w, activation=activation).double() - a * up).abs() <= limit).all())


@pytest.mark.parametrize("M", [1, 4, 8])
def test_infinities_and_nan_stay_in_their_rows(M):
    from spyinfer_amd.kernels import ops
    dev = require_gpu()
    x, w = torch.ones((M, 1100), device=dev), torch.ones((1500, 1100), device=dev)
    x[M - 1, 1099], w[1499, 7], w[3, 1098], w[1030] = float("inf"), float("nan"), float("-inf"), 0.0
    want = x @ w.t()
    out = ops.linear(x, w)
    assert torch.equal(out.isnan(), want.isnan()) and torch.equal(out[~want.isnan()], want[~want.isnan()])
