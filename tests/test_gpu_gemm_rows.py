"""Products of many rows from the tiled copy (csrc/gemm_rows.hip): one turn of K, two, an odd number of them, parts of uneven length,
every number of row tiles, a last tile of rows that reaches back, columns that are no multiple of a block's; and the norm that sums a
product's parts; against float64."""
import pytest
import torch

from tests.gpu_util import close, require_gpu

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M,N,K,tiles,parts", [(65, 272, 128, 4, 1), (128, 256, 256, 8, 2), (200, 1040, 384, 7, 3), (131, 512, 640, 5, 2), (193, 48, 1280, 6, 4),
                                               (112, 768, 896, 7, 7), (500, 256, 512, 8, 1)])
def test_parts(M, N, K, tiles, parts, monkeypatch):
    from spyinfer_amd.kernels import ops
    monkeypatch.setattr(ops, "rows_product_parts", lambda *size: (tiles, parts))
    dev = require_gpu()
    g = torch.Generator().manual_seed(M + N)
    x, w = torch.randn((M, K), generator=g).bfloat16(), (torch.randn((N, K), generator=g) * K ** -0.5).bfloat16()
    wd = w.to(dev)
    out = ops.linear_parts(x.to(dev), wd, ops.tile_weight(wd))
    assert isinstance(out, ops.ProductParts) and tuple(out.parts.shape) == (parts, M, N)
    # exact products of bfloat16 values, K float32 sums of terms of size K^-1/2: an error of some 2^-24 sqrt(K) terms' sizes
    bounds = [K // 128 * p // parts * 128 for p in range(parts + 1)]
    for p, (a, b) in enumerate(zip(bounds, bounds[1:])):
        ref = x[:, a:b].double() @ w[:, a:b].double().T
        assert float((out.parts[p].cpu().double() - ref).abs().max()) < 1e-5


@pytest.mark.parametrize("M,N,K,tiles", [(65, 272, 128, 4), (200, 1040, 384, 7), (131, 512, 640, 5), (193, 48, 1024, 6), (300, 256, 256, 8)])
def test_stored(M, N, K, tiles, monkeypatch):
    from spyinfer_amd.kernels import ops
    monkeypatch.setattr(ops, "rows_product_stored", lambda *size: tiles)
    dev = require_gpu()
    g = torch.Generator().manual_seed(M + N)
    x, w = torch.randn((M, K), generator=g).bfloat16(), (torch.randn((N, K), generator=g) * K ** -0.5).bfloat16()
    wd = w.to(dev)
    close(ops.linear(x.to(dev), wd, tiled=ops.tile_weight(wd)), x.double() @ w.double().T, torch.bfloat16, what="product of many rows")


@pytest.mark.parametrize("M,N,K,parts", [(17, 64, 32, 1), (65, 100, 132, 2), (64, 1000, 2048, 12), (130, 66, 1000, 5), (200, 384, 612, 3)])
def test_float32_parts(M, N, K, parts, monkeypatch):
    from spyinfer_amd.kernels import ops
    monkeypatch.setattr(ops, "f32_product_parts", lambda *size: parts)
    dev = require_gpu()
    g = torch.Generator().manual_seed(M + N)
    x, w = torch.randn((M, K), generator=g), torch.randn((N, K), generator=g) * K ** -0.5
    out = ops.linear_parts(x.to(dev), w.to(dev))
    assert isinstance(out, ops.ProductParts) and tuple(out.parts.shape) == (parts, M, N)
    steps = -(-K // 32)
    bounds = [min(K, steps * p // parts * 32) for p in range(parts + 1)]
    for p, (a, b) in enumerate(zip(bounds, bounds[1:])):
        ref = x[:, a:b].double() @ w[:, a:b].double().T
        assert float((out.parts[p].cpu().double() - ref).abs().max()) < 1e-5           # (as above)


@pytest.mark.parametrize("activation", ["silu", "gelu_tanh"])
@pytest.mark.parametrize("M,I,K,tiles", [(65, 128, 128, 4), (200, 144, 256, 7), (131, 16, 384, 5), (193, 1040, 640, 6), (300, 384, 1152, 8)])
def test_gated(M, I, K, tiles, activation, monkeypatch):
    from spyinfer_amd.kernels import ops
    monkeypatch.setattr(ops, "rows_product_gated", lambda *size: tiles)
    dev = require_gpu()
    g = torch.Generator().manual_seed(M + I)
    x, w = torch.randn((M, K), generator=g).bfloat16(), (torch.randn((2 * I, K), generator=g) * K ** -0.5).bfloat16()
    wd = w.to(dev)
    out = ops.linear_swiglu(x.to(dev), wd, ops.tile_weight(wd), activation=activation)
    h = x.double() @ w.double().T
    act = torch.nn.functional.silu if activation == "silu" else lambda z: torch.nn.functional.gelu(z, approximate="tanh")
    close(out, act(h[:, :I]) * h[:, I:], torch.bfloat16, what="gated product of many rows")


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("T,H,parts", [(65, 64, 1), (70, 516, 3), (130, 2560, 6), (66, 8192, 2)])
def test_norm_of_a_sum_of_parts(T, H, parts, dtype):
    from spyinfer_amd.kernels import ops
    dev = require_gpu()
    g = torch.Generator().manual_seed(T + H)
    resid, y = torch.randn((T, H), generator=g), torch.randn((parts, T, H), generator=g)
    w = torch.randn((H,), generator=g).to(dtype)
    rows = torch.tensor([T - 1, 0, 7], dtype=torch.int32)
    total = resid.double() + y.double().sum(0)
    ref = total / torch.sqrt((total * total).mean(-1, keepdim=True) + 1e-6) * w.double()
    stream = resid.to(dev)
    some = ops.add_parts_rms_norm(stream, ops.ProductParts(y.to(dev)), w.to(dev), 1e-6, dtype, rows.to(dev))
    assert torch.equal(stream.cpu(), resid)                       # (picked rows: the stream stays as it is)
    close(some, ref[rows.long()], dtype, what="picked rows")
    close(ops.add_parts_rms_norm(stream, ops.ProductParts(y.to(dev)), w.to(dev), 1e-6, dtype), ref, dtype, what="normed sum")
    close(stream, total, torch.float32, what="the stream")


def test_rules_of_steps_that_are_replayed(tmp_path, monkeypatch):
    """140 requests decoding: the step before the capture and the capture ask the rule alike, for a step whose launches the host pays once;
    a prompt and steps that no graph will hold ask for steps launched one by one."""
    from spyinfer_amd.engine.batch import StepEntry
    from spyinfer_amd.engine.runner import ModelRunner, load_model
    from spyinfer_amd.kernels import ops
    from spyinfer_amd.weights import write_random_model
    from tests.configs import INIT, TINY_E
    dev = require_gpu()
    asked = []
    monkeypatch.setattr(ops, "rows_product_stored", lambda M, N, K, replayed: asked.append(replayed) or 0)
    folder = write_random_model(str(tmp_path / "model"), TINY_E, seed=3, dtype=torch.bfloat16, **INIT)
    runner = ModelRunner(load_model(folder, "bfloat16", dev), "bfloat16", dev, 16, 200, 140, enforce_eager=False, max_model_len=32)
    live = [runner.manager.admit("r%d" % i) for i in range(140)]

    def step(tokens):
        asked.clear()
        for rc, t in zip(live, tokens):
            runner.manager.reserve(rc, len(t))
        return runner.step([StepEntry(rc, t, (len(t) - 1,)) for rc, t in zip(live, tokens)]).clone()

    step([[i % 500, 7] for i in range(140)])
    assert asked and not any(asked)
    first = step([[i % 400] for i in range(140)])
    assert asked and all(asked)
    outs = []
    for _ in range(3):
        for rc in live:
            assert runner.manager.rewind(rc, 2)
        outs.append(step([[i % 400] for i in range(140)]))
        assert all(asked)
    assert runner.graph_replays == 3 and all(torch.equal(o, first) for o in outs)
    runner.max_graphs = 1
    live = live[:139]
    step([[5]] * 139)
    assert asked and not any(asked)


def test_library_products_of_replayed_steps(monkeypatch):
    from spyinfer_amd.kernels import ops
    dev = require_gpu()
    x, w = torch.randn((130, 1024), device=dev).bfloat16(), torch.randn((4096, 1024), device=dev).bfloat16()
    tiled = ops.tile_weight(w)
    with ops.replayed_step():
        assert torch.equal(ops.linear(x, w, tiled=tiled), x @ w.t())
        monkeypatch.setattr(ops.TiledOnly, "rows", lambda self: pytest.fail("rows copied for the library's product"))
        close(ops.linear(x, ops.TiledOnly(tiled)), x.double() @ w.double().t(), torch.bfloat16, what="product of a matrix kept in tiles only")


@pytest.mark.parametrize("form", ["parts", "stored", "gated"])
def test_infinities_and_nan_stay_in_their_rows(form, monkeypatch):
    """A row with NaN and one with infinities, in the rows that the last tile shares with the one before; and a row of the matrix."""
    from spyinfer_amd.kernels import ops
    dev = require_gpu()
    M, N, K = 200, 1056, 384
    monkeypatch.setattr(ops, "rows_product_parts", lambda *size: (7, 3))
    monkeypatch.setattr(ops, "rows_product_stored", lambda *size: 7)
    monkeypatch.setattr(ops, "rows_product_gated", lambda *size: 7)
    g = torch.Generator().manual_seed(6)
    x, w = torch.randn((M, K), generator=g).bfloat16(), torch.randn((N, K), generator=g).bfloat16()
    x[100, 3], x[M - 1, 70], w[N - 1, 200] = float("nan"), float("inf"), float("nan")
    x, w = x.to(dev), w.to(dev)
    ref = x.float() @ w.float().t()
    if form == "parts":
        got = ops.linear_parts(x, w, ops.tile_weight(w)).resolve()
    elif form == "stored":
        got = ops.linear(x, w, tiled=ops.tile_weight(w))
    else:
        got = ops.linear_swiglu(x, w, ops.tile_weight(w))
        ref = ops.swiglu(ref)                                        # (its activation as it is for infinite values)
    assert torch.equal(got.isnan(), ref.isnan()) and torch.equal(got.isinf(), ref.isinf())
    some = torch.arange(M, device=dev)[~ref[:, 0].isnan() & ~ref[:, 0].isinf()]
    assert len(some) == M - 2
    close(got[some, :-1], ref[some, :-1], torch.bfloat16, scale=2.0, what="the other rows")


def test_operands_off_16_bytes():
    """Views that begin between two 16-byte pieces: the kernels that take no such operand are passed by."""
    from spyinfer_amd.kernels import ops
    dev = require_gpu()

    def off(t, n):
        buf = torch.empty((t.numel() + 8,), dtype=t.dtype, device=dev)[n:n + t.numel()].view(t.shape)
        return buf.copy_(t)

    g = torch.Generator().manual_seed(8)
    x, w, small = torch.randn((600, 1024), generator=g), torch.randn((4096, 1024), generator=g) / 32, torch.randn((1024, 2048), generator=g) / 45
    xb, wb = off(x.bfloat16(), 4), w.bfloat16().to(dev)
    tiled, ref = ops.tile_weight(wb), x.bfloat16().double() @ w.bfloat16().double().t()
    assert xb.data_ptr() % 16 and ops.rows_product_stored(600, 4096, 1024) and ops.rows_product_gated(600, 4096, 1024, True)
    close(ops.linear(xb, wb, tiled=tiled), ref, torch.bfloat16, what="rows off 16 bytes")
    out = off(torch.zeros((600, 4096)).bfloat16(), 4)
    assert ops.linear(xb.clone(), wb, tiled=tiled, out=out) is out
    close(out, ref, torch.bfloat16, what="a result off 16 bytes")
    close(ops.linear_swiglu(xb, wb, tiled), torch.nn.functional.silu(ref[:, :2048]) * ref[:, 2048:], torch.bfloat16, what="gated, rows off 16 bytes")
    sb, xs = small.bfloat16().to(dev), torch.randn((200, 2048), generator=g)
    assert ops.rows_product_parts(200, 1024, 2048)
    y = ops.linear_parts(off(xs.bfloat16(), 4), sb, ops.tile_weight(sb))
    close(y, xs.bfloat16().double() @ small.bfloat16().double().t(), torch.bfloat16, what="parts, rows off 16 bytes")
    assert ops.f32_product_parts(200, 1024, 2048)
    for x32, w32 in ((off(xs, 1), small.to(dev)), (xs.to(dev), off(small, 1))):
        close(ops.linear_parts(x32, w32), xs.double() @ small.double().t(), torch.float32, what="float32 off 16 bytes")
    h = xs[:3].double() @ small.double().t()
    close(ops.linear_swiglu(off(xs[:3], 1), small.to(dev)), torch.nn.functional.silu(h[:, :512]) * h[:, 512:], torch.float32, what="gated float32 off 16 bytes")
