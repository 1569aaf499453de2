"""Float32 products whose values are cut into bfloat16 parts (csrc/gemm_f32_split.hip) against 64 bits: both tiles at their edges, one step
of 32 of K to more than the loads run ahead, parts of uneven length, the gated product, values that cannot be cut."""
import pytest
import torch

from tests.gpu_util import require_gpu

pytestmark = pytest.mark.gpu

# (M, N, K): the small tile, the large one, columns that are multiples of nothing
SHAPES = [(33, 8192, 32), (64, 8130, 64), (65, 4097, 96), (129, 5441, 128), (130, 8190, 160), (257, 2052, 192), (611, 1030, 224), (385, 1283, 1024),
          (640, 5377, 288), (1030, 4100, 256), (300, 1700, 4160)]


def operands(M, N, K, dev):
    g = torch.Generator().manual_seed(M + 3 * N + 7 * K)
    # (values of many sizes: each by a power of two of its own)
    x, w = (torch.randn((n, K), generator=g) * torch.exp2(torch.randint(-8, 8, (n, K), generator=g).float()) for n in (M, N))
    return x.to(dev), w.to(dev)


def bound(x, w):
    # what is left out of a product of two values is at most 2^-24 of it (each middle part at most 2^-8 of its value, each low part 2^-17); an
    # instruction, sixteen of K, rounds four times at most, a chain has 2048 of K at most before the sums' sums
    K = x.shape[1]
    return (1 + 4 * -(-min(K, 2048) // 16) + K / 512 + 8) * 2.0 ** -24 * (x.double().abs() @ w.double().abs().t())


def close_in_norm(out, want):
    # 1.9e-7 to 3.0e-7 with all of the six products of parts; without one of the three smallest 1e-6 and more
    assert float((out.double() - want).norm() / want.norm()) < 4.5e-7


@pytest.mark.parametrize("M,N,K", SHAPES)
def test_product(M, N, K):
    from spyinfer_amd.kernels import ops
    dev = require_gpu()
    assert ops.f32_rows_split(M, N, K)
    x, w = operands(M, N, K, dev)
    held = torch.full((M * N + 4096,), float("nan"), device=dev)          # what lies behind the result stays as it is
    out = ops.linear(x, w, out=held[:M * N].view(M, N))
    want = x.double() @ w.double().t()
    assert bool(((out.double() - want).abs() <= bound(x, w)).all())
    close_in_norm(out, want)
    assert bool(held[M * N:].isnan().all())
    w = w.bfloat16().float()                                             # (the products of a matrix that a bfloat16 checkpoint gave)
    close_in_norm(ops.linear(x, w), x.double() @ w.double().t())


@pytest.mark.parametrize("M,N,K,parts", [(33, 70, 64, 2), (129, 130, 416, 3), (200, 2048, 1056, 12), (611, 1030, 1120, 5), (300, 3000, 2048, 2)])
def test_parts(M, N, K, parts, monkeypatch):
    from spyinfer_amd.kernels import ops
    dev = require_gpu()
    monkeypatch.setattr(ops, "f32_product_parts", lambda *size: parts)
    x, w = operands(M, N, K, dev)
    out = ops.linear_parts(x, w).parts
    for p in range(parts):
        a, b = K // 32 * p // parts * 32, K // 32 * (p + 1) // parts * 32
        close_in_norm(out[p], x[:, a:b].double() @ w[:, a:b].double().t())
        assert bool(((out[p].double() - x[:, a:b].double() @ w[:, a:b].double().t()).abs() <= bound(x[:, a:b], w[:, a:b])).all())


@pytest.mark.parametrize("activation", ["silu", "gelu_tanh"])
@pytest.mark.parametrize("M,I,K", [(33, 4096, 32), (65, 2050, 160), (200, 6111, 96), (611, 3072, 1024)])
def test_gated(M, I, K, activation):
    from spyinfer_amd.kernels import ops
    dev = require_gpu()
    x, w = operands(M, 2 * I, K, dev)
    x, w = x / 16, w / (16 * K ** 0.5)
    h, err = x.double() @ w.double().t(), bound(x, w)
    act = torch.nn.functional.silu if activation == "silu" else lambda z: torch.nn.functional.gelu(z, approximate="tanh")
    out = ops.linear_swiglu(x, w, activation=activation)
    a, up = act(h[:, :I]), h[:, I:]
    # (both activations' slopes are below 1.13; the activation itself is a handful of roundings)
    limit = 1.13 * err[:, :I] * (up.abs() + err[:, I:]) + a.abs() * err[:, I:] + 16 * 2.0 ** -24 * (h[:, :I] * up).abs() + 1e-30
    assert bool(((out.double() - a * up).abs() <= limit).all())
    # (both halves' errors meet, and a gate of some size passes on several times its own)
    assert float((out.double() - a * up).norm() / (a * up).norm()) < 1.2e-6


@pytest.mark.parametrize("M,N", [(65, 4100), (611, 4100)])
@pytest.mark.parametrize("how", ["product", "gated", "parts"])
def test_every_product_of_parts(M, N, how, monkeypatch):
    """One number of 96 is set in each row of both operands, and the products have at most 24 bits: every result is exact, and each of the six
    products of parts decides some of them."""
    from spyinfer_amd.kernels import ops
    dev, K = require_gpu(), 96
    h, m, l = 1.0, 2.0 ** -8 * 0.75, 2.0 ** -17 * 0.625                  # (one part each: below half of the last place of the one before)
    pairs = [(h + m + l, h), (h, h + m + l), (h + m, h + m), (h + l, 3 * h), (-5 * h, h + l), (m + l, 3 * h), (7 * h, -(m + l)), (m, m), (h - m, h + m), (l, h)]
    x, w = torch.zeros((M, K), dtype=torch.float64), torch.zeros((N, K), dtype=torch.float64)
    for i in range(M):
        x[i, i % 80] = pairs[i % 10][0]
    for j in range(N):
        for k in range(80):
            if (j + k) % 3 == 0:
                w[j, k] = pairs[k % 10][1]
    x, w = x.to(dev), w.to(dev)
    want = x @ w.t()
    assert torch.equal(want.float().double(), want) and torch.equal(x.float().double(), x) and torch.equal(w.float().double(), w)
    x, w = x.float(), w.float()
    if how == "product":
        assert torch.equal(ops.linear(x, w), want.float())
    elif how == "parts":
        monkeypatch.setattr(ops, "f32_product_parts", lambda *size: 3)
        assert torch.equal(ops.linear_parts(x, w).parts.sum(0), want.float())
    else:
        # gates of 64 pass the other half on times 64, but for the last place
        w[:N // 2], x[:, 95], w[:N // 2, 95] = 0.0, 64.0, 1.0
        out, want = ops.linear_swiglu(x, w), 64 * want[:, N // 2:]
        assert bool(((out.double() - want).abs() <= 2.0 ** -23 * want.abs()).all())


@pytest.mark.parametrize("M,N", [(65, 5000), (611, 5000)])
@pytest.mark.parametrize("size", [-108, -112, -118, -124, -130])
@pytest.mark.parametrize("side", ["rows", "matrix"])
def test_small_numbers(M, N, size, side):
    """Numbers whose low parts are below bfloat16's smallest one, beside large ones: results are as exact as others', and the rows and columns
    without such numbers are bit for bit what they are without them."""
    from spyinfer_amd.kernels import ops
    dev, K = require_gpu(), 544
    g = torch.Generator().manual_seed(M + N + size)
    x, w = torch.randn((M, K), generator=g).to(dev), (torch.randn((N, K), generator=g) * 2.0 ** 20).to(dev)
    before = ops.linear(x, w)
    a, b = (x, w) if side == "rows" else (w, x)
    a[3::7, 33] = (1 + torch.rand((a[3::7].shape[0],), generator=g)).to(dev).double().mul(2.0 ** size).float()
    a[5] = (torch.randn((K,), generator=g)).to(dev).double().mul(2.0 ** size).float()
    out, want = ops.linear(x, w), x.double() @ w.double().t()
    # (products themselves are numbers of more than 2^-126 + 24, but for those of 2^-130)
    assert bool(((out.double() - want).abs() <= bound(x, w) + 2.0 ** -149 * K).all())
    if size > -130:
        close_in_norm(*((out[5], want[5]) if side == "rows" else (out[:, 5], want[:, 5])))
    untouched = torch.ones(a.shape[0], dtype=torch.bool)
    untouched[3::7], untouched[5] = False, False
    assert torch.equal(*((t[untouched] if side == "rows" else t[:, untouched]) for t in (out, before)))


@pytest.mark.parametrize("M,N", [(65, 5000), (600, 5000)])
@pytest.mark.parametrize("gated", [False, True])
def test_values_that_cannot_be_cut(M, N, gated):
    """Infinities, NaN and values that bfloat16 rounds to infinity: the rows and columns they stand in are what float32 arithmetic makes of
    them, all others as ever."""
    from spyinfer_amd.kernels import ops
    dev = require_gpu()
    x, w = torch.ones((M, 96), device=dev), torch.ones((N, 96), device=dev)
    x[M - 1, 3], x[M - 2, 70], x[5, 1] = float("inf"), float("nan"), 3.4e38
    w[N - 1, 7], w[0, 95], w[64] = float("nan"), float("-inf"), 1e-38
    x[5, 2], w[9, 1] = -3.4e38, -1.0
    want = (x.double() @ w.double().t()).float()
    if gated:
        out, want = ops.linear_swiglu(x, w), ops.swiglu(want)          # (the activation of infinities is the activation pass's)
    else:
        out = ops.linear(x, w)
    finite = want.isfinite()
    assert torch.equal(out.isnan(), want.isnan()) and torch.equal(out[want.isinf()], want[want.isinf()])
    # (96 values of up to 3.4e38 that cancel but for a rounding of the largest; a gated one's other half is at most as large again)
    assert bool(((out - want).abs() <= 96 * 2.0 ** -24 * (x.abs().double() @ w.abs().double().t()).float()[:, :want.shape[1]].clamp(min=1.0))[finite].all())
    if not gated:
        plain = torch.ones(M, dtype=torch.bool)
        plain[[5, M - 1, M - 2]] = False
        assert bool(((out - want).abs() <= 96 * 2.0 ** -24 * want.abs())[plain][:, 64].all())         # the column of 1e-38, relatively


@pytest.mark.parametrize("M,N,K", [(65, 4100, 32), (130, 5441, 160), (611, 4096, 1024), (300, 1700, 4160)])
@pytest.mark.parametrize("where", ["nowhere", "first", "inside", "last"])
def test_matrices_of_bfloat16_values(M, N, K, where):
    """A matrix whose values are bfloat16 numbers, but for one of a row: the other rows' results are those of the matrix without it, bit for
    bit, whichever way their tiles went."""
    from spyinfer_amd.kernels import ops
    dev = require_gpu()
    x, w = operands(M, N, K, dev)
    w = w.bfloat16().float()
    whole = ops.linear(x, w)
    assert bool(((whole.double() - x.double() @ w.double().t()).abs() <= bound(x, w)).all())
    if where != "nowhere":
        w[N - 1, {"first": 0, "inside": K // 2, "last": K - 1}[where]] = 1.0 + 2.0 ** -20
    out = ops.linear(x, w)
    assert torch.equal(out[:, :N - 1], whole[:, :N - 1])
    assert bool(((out.double() - x.double() @ w.double().t()).abs() <= bound(x, w)).all())
    parts = ops.linear_swiglu(x, w[:N // 2 * 2].contiguous())
    g = x.double() @ w.double().t()
    a, up = torch.nn.functional.silu(g[:, :N // 2]), g[:, N // 2:N // 2 * 2]
    assert float((parts.double() - a * up).norm() / (a * up).norm()) < 1e-5


@pytest.mark.parametrize("M,N,K", [(65, 4100, 1184), (611, 4096, 1120)])
@pytest.mark.parametrize("gated", [False, True])
def test_the_step_of_the_first_value_that_is_no_bfloat16_number(M, N, K, gated):
    """A block goes on from the step in which it meets such a value: the other rows of the matrix have the bits that they have without it,
    whichever of the steps it is, and its own row has the product in full."""
    from spyinfer_amd.kernels import ops
    dev = require_gpu()
    x, w = operands(M, N, K, dev)
    w = w.bfloat16().float()
    product = ops.linear_swiglu if gated else ops.linear
    whole, row = product(x, w), N // 2 - 3
    others = torch.arange(N // 2 if gated else N, device=dev) != row
    for k in range(31, K, 32):
        kept, w[row, k] = float(w[row, k]), 0.7 + 2.0 ** -20
        out = product(x, w)
        assert torch.equal(out[:, others], whole[:, others]), k
        if not gated:
            assert bool(((out[:, row].double() - x.double() @ w[row].double()).abs() <= bound(x, w[row:row + 1])[:, 0]).all()), k
        w[row, k] = kept


@pytest.mark.parametrize("M,N", [(65, 5000), (611, 5000)])
@pytest.mark.parametrize("gated", [False, True])
def test_neighbours_of_values_that_cannot_be_cut(M, N, gated):
    """Rows and columns beside an infinity, a NaN or a value beyond bfloat16's range are bit for bit what they are without it; and the results
    of a row with such a value that a zero of the matrix takes away are as exact as others."""
    from spyinfer_amd.kernels import ops
    dev, K = require_gpu(), 2080
    g = torch.Generator().manual_seed(M + N)
    x, w = torch.randn((M, K), generator=g).to(dev), (torch.randn((N, K), generator=g) * K ** -0.5).to(dev)
    w[:, 1030] = 0.0
    product = ops.linear_swiglu if gated else ops.linear
    before = product(x, w)
    y, v = x.clone(), w.clone()
    y[3, 77], y[M - 1, 2079], y[40, 1030] = float("inf"), float("nan"), 3.4e38
    v[N // 2 + 9, 5], v[20, 1000] = float("-inf"), float("nan")
    out = product(y, v)
    rows, columns = torch.ones(M, dtype=torch.bool), torch.ones(out.shape[1], dtype=torch.bool)
    rows[[3, 40, M - 1]], columns[[9 if gated else N // 2 + 9, 20]] = False, False
    assert torch.equal(out[rows][:, columns], before[rows][:, columns])
    if not gated:
        want = x[40].double() @ w.double().t()
        columns = columns.to(dev)
        # (the chains of float32 instructions end every 256 of K: 2.9e-7 as gemm_f32.hip has it; one chain over all of K has 8e-7)
        assert float((out[40].double() - want)[columns].norm() / want[columns].norm()) < 4e-7
