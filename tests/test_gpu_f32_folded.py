"""The float32 products of a few rows with the norm before them, or the sum into the stream behind them, folded in (csrc/gemm_f32.hip)."""
import pytest
import torch

from spyinfer_amd.kernels import ops

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
EPS = 1e-6

# (rows, columns, K): every number of rows a block is built for and between them; columns beside and at the sizes of a block and at the lines of
# the rule for blocks; K below a lane's piece of a wave, a rest behind whole chunks of 256, a rest of rounds, and whole rounds
SIZES = [(1, 1, 4), (1, 1000, 1024), (1, 4097, 2052), (2, 7, 260), (2, 1025, 1024), (3, 1023, 516), (4, 1024, 3072), (4, 2050, 2048), (4, 8193, 256),
         (5, 30, 1024), (6, 4095, 768), (8, 4096, 1024), (8, 1024, 2048), (8, 9, 5124)]


def _bound(terms, K):
    # every sum has at most K / 256 pieces of 4 in a lane, 8 additions over lanes and 32 over waves, and 8 roundings for norm, scale and sum
    return (K / 64 + 48) * 2.0 ** -23 * terms


def _case(M, N, K, seed, factor=1):
    gen = torch.Generator().manual_seed(seed)
    x = torch.randn((M, K), generator=gen) * torch.logspace(-3, 3, M)[:, None]
    w = torch.randn((factor * N, K), generator=gen) * K ** -0.5
    g = 1.0 + 0.2 * torch.randn((K,), generator=gen)
    return x, w, g


def _normed(x, g):
    x = x.double()
    return x / torch.sqrt((x * x).mean(dim=1, keepdim=True) + EPS) * g.double()


def _scaled(x, g, parts):
    """The input as a product into the stream leaves it, its squares in ``parts`` parts."""
    rows = 1 << (x.shape[0] - 1).bit_length()
    ss = torch.zeros((parts, rows))
    squares = torch.nn.functional.pad(x * x, (0, -x.shape[1] % parts)).reshape(x.shape[0], -1, parts).sum(dim=1)
    ss[:, :x.shape[0]] = squares.t()
    return ops.ScaledF32((x * g).to(DEV), ss.to(DEV), EPS)


# (one part of the squares, fewer than a block has threads, and more than its threads ask for ahead)
@pytest.mark.parametrize("parts", [1, 37, 2500])
@pytest.mark.parametrize("M,N,K", SIZES)
def test_products_of_the_normed_stream(M, N, K, parts):
    x, w, g = _case(M, N, K, M + N + K)
    got = ops.scaled_f32_linear(_scaled(x, g, parts), w.to(DEV)).cpu().double()
    n = _normed(x, g)
    assert bool(((got - n @ w.double().t()).abs() <= _bound(n.abs() @ w.double().abs().t(), K)).all())


@pytest.mark.parametrize("activation", ["silu", "gelu_tanh"])
@pytest.mark.parametrize("M,N,K", SIZES)
def test_gated_products_of_the_normed_stream(M, N, K, activation):
    x, w, g = _case(M, N, K, M + N + K + 1, 2)
    got = ops.scaled_f32_swiglu(_scaled(x, g, 64), w.to(DEV), activation).cpu().double()
    n = _normed(x, g)
    z, u = n @ w.double()[:N].t(), n @ w.double()[N:].t()
    act = torch.nn.functional.silu if activation == "silu" else (lambda t: torch.nn.functional.gelu(t, approximate="tanh"))
    bz, bu = _bound(n.abs() @ w.double()[:N].abs().t(), K), _bound(n.abs() @ w.double()[N:].abs().t(), K)
    # (the activations' slope is at most 1.13, their value at most |z|; their own functions are right to a few parts in 2^23)
    assert bool(((got - act(z) * u).abs() <= 1.13 * bz * (u.abs() + bu) + z.abs() * bu + 16 * 2.0 ** -23 * ((z * u).abs() + u.abs())).all())


@pytest.mark.parametrize("M,N,K", SIZES)
def test_sums_into_the_stream(M, N, K):
    x, w, g = _case(M, N, K, M + N + K + 2)
    h = torch.randn((M, N), generator=torch.Generator().manual_seed(5))
    stream, after_w = h.to(DEV), 1.0 + 0.3 * torch.randn((N,), generator=torch.Generator().manual_seed(6))
    after = ops.f32_linear_residual(x.to(DEV), w.to(DEV), stream, after_w.to(DEV), EPS)
    want = h.double() + x.double() @ w.double().t()
    assert bool(((stream.cpu().double() - want).abs() <= _bound(x.double().abs() @ w.double().abs().t(), K) + 2.0 ** -23 * want.abs()).all())
    assert torch.equal(after.xw, stream * after_w.to(DEV))
    squares = after.ss_parts.cpu().double().sum(dim=0)
    want = (stream.cpu().double() ** 2).sum(dim=1)
    assert bool(((squares[:M] - want).abs() <= 8 * 2.0 ** -23 * want).all()) and bool((squares[M:] == 0).all())       # (a part: up to 8 columns)


def test_what_is_refused():
    x, w, g = _case(9, 8, 256, 1)
    with pytest.raises(ops.KernelError):
        ops.scaled_f32_linear(_scaled(x, g, 2), w.to(DEV))
    with pytest.raises(ops.KernelError):
        ops.scaled_f32_linear(_scaled(x[:4, :128], g[:128], 2), w.to(DEV))
    with pytest.raises(ops.KernelError):
        ops.f32_linear_residual(x.to(DEV), w.to(DEV), torch.zeros((9, 8), device=DEV), torch.ones(8, device=DEV), EPS)


@pytest.mark.parametrize("requests", [1, 4, 8])
def test_steps_with_and_without_folded_norms(requests, tmp_path):
    """Decoding with the norms folded in and by kernels of their own, eagerly and from graphs: the same logits within what float32 sums of
    another order differ by (2e-5 of a logit's size of a few; 12 roundings a layer of 1e-7 each and their growth over the layers)."""
    from spyinfer_amd.engine.batch import StepEntry
    from spyinfer_amd.engine.runner import ModelRunner, load_model
    from spyinfer_amd.weights import write_random_model
    from tests.configs import INIT, TINY_D
    model = load_model(write_random_model(str(tmp_path / "m"), TINY_D, 63, torch.bfloat16, **INIT), "float32", DEV)
    gen = torch.Generator().manual_seed(3)
    prompts = [torch.randint(0, 400, (5 + 9 * i,), generator=gen).tolist() for i in range(requests)]
    real, runs, calls = ops.f32_linear_residual, [], []
    for folded, eager in ((True, True), (True, False), (False, True)):
        ops.FUSED_DECODE, n = folded, [0]
        ops.f32_linear_residual = lambda *a, **k: (n.__setitem__(0, n[0] + 1), real(*a, **k))[1]
        try:
            runner = ModelRunner(model, "float32", DEV, 16, 96, requests, enforce_eager=eager, max_model_len=320)
            caches = [runner.manager.admit(i) for i in range(requests)]
            for c, p in zip(caches, prompts):
                runner.manager.reserve(c, len(p))
            runner.step([StepEntry(c, p, []) for c, p in zip(caches, prompts)])
            tokens, outs = torch.Generator().manual_seed(4), []
            for _ in range(6):
                step = torch.randint(0, 400, (requests,), generator=tokens).tolist()
                for c in caches:
                    runner.manager.reserve(c, 1)
                outs.append(runner.step([StepEntry(c, [t], [0]) for c, t in zip(caches, step)]).cpu().clone())
            runs.append(outs)
            calls.append(n[0])
        finally:
            ops.FUSED_DECODE, ops.f32_linear_residual = True, real
    assert calls[0] > 0 and calls[2] == 0
    for a, b, c in zip(*runs):
        assert torch.equal(a, b) and torch.allclose(a, c, rtol=2e-5, atol=2e-5), (a - c).abs().max()


# (query heads, kv heads, head size, page, keys before the step's token by request, window, head norms, rotation): no key before, the edges of blocks of
# 16 keys and of pages, one part of the keys and many, more parts than blocks, a window that ends with the new key alone
RAW_CASES = [(16, 8, 128, 16, [0, 1, 15, 16, 17, 500], None, True, True), (8, 1, 128, 32, [31, 32, 33, 1300], None, True, True), (4, 4, 64, 16, [700], None, False, True),
             (32, 2, 64, 64, [63, 64, 200, 5, 129], None, True, False), (16, 8, 128, 16, [40, 300, 16, 2], 1, True, True), (6, 2, 128, 48, [47, 48, 95, 333], 50, True, True)]


@pytest.mark.parametrize("case", range(len(RAW_CASES)))
def test_attention_taking_the_raw_product(case):
    """Single tokens: the attention norms, rotates and stores by itself.  The new tokens' places hold NaN before the call; the rest of the cache stays as
    it was.  Reference: the plain attention in float64 over the normed and rotated rows."""
    from spyinfer_amd.parts.rotary import RotaryEmbedding
    from tests.test_gpu_kernels import make_attention_case, plain_paged_attention, plain_qk
    n_q, n_kv, d, P, cached, window, norm, rotate = RAW_CASES[case]
    f32, T = torch.float32, len(cached)
    _q, kc, vc, bt, te, ps, meta = make_attention_case(f32, DEV, n_q, n_kv, d, P, [(a, 1) for a in cached], seed=70 + case, window=window)
    gen = torch.Generator().manual_seed(case)
    qkv = torch.randn((T, (n_q + 2 * n_kv) * d), generator=gen)
    qw, kw = ((1 + 0.2 * torch.randn((d,), generator=gen)) if norm else None for _ in range(2))
    rope = RotaryEmbedding(d, 23456.0, d)
    rope.prepare(DEV, 2100)
    rq, rk, rv = plain_qk(qkv, n_q, n_kv, d, qw, kw, 1e-6, 23456.0, d if rotate else 0, torch.tensor(cached, dtype=torch.int32))
    kc_ref, vc_ref, new = kc.clone(), vc.clone(), torch.zeros(kc.shape[:3], dtype=torch.bool)
    kc_dev, vc_dev = kc.clone(), vc.clone()
    for s, a in enumerate(cached):
        page = bt[s][a // P]
        kc_ref[page, :, a % P, :], vc_ref[page, :, :, a % P] = rk[s].to(f32), rv[s].to(f32)
        kc_dev[page, :, a % P, :] = vc_dev[page, :, :, a % P] = float("nan")
        new[page, :, a % P] = True
    scale = d ** -0.5
    ref = plain_paged_attention(rq.reshape(T, n_q * d).to(f32), kc_ref, vc_ref, P, bt, te, ps, n_q, n_kv, d, scale, window).double()
    on = lambda t: None if t is None else t.to(DEV)
    assert ops.fused_attention_ok(f32, meta, n_q, n_kv, d, P, d if rotate else 0, on(qw), on(kw))
    raw = ops.RawQKV(on(qkv), on(qw), on(kw), 1e-6, rope.cos if rotate else None, rope.sin if rotate else None, True)
    # A score has d products of sizes up to 10 times 10 over sqrt(d), each rounded, and the rotation's table 2^-24 of an angle of up to 1300: 1e-4 of a
    # score, and as much of a weight; values are of size one
    near = lambda a, b: torch.allclose(a.cpu().double(), b.double(), rtol=1e-4, atol=1e-4)
    k1, v1 = on(kc_dev), on(vc_dev)
    out = ops.paged_attention(None, k1, v1, P, meta, n_q, n_kv, d, scale, window, raw)
    assert near(out, ref), (out.cpu().double() - ref).abs().max()
    same = lambda a, b: torch.equal(torch.nan_to_num(a.cpu(), nan=-77.0), torch.nan_to_num(b, nan=-77.0))
    assert same(v1, vc_ref) and same(k1.cpu()[~new], kc_ref[~new]) and near(k1.cpu()[new], kc_ref[new])
    # nothing stored, the new place read from the cache
    k2, v2 = on(kc_ref), on(vc_ref)
    raw.store = False
    out = ops.paged_attention(None, k2, v2, P, meta, n_q, n_kv, d, scale, window, raw)
    assert near(out, ref) and same(k2, kc_ref) and same(v2, vc_ref)


@pytest.mark.parametrize("hidden,inner,rows", [(512, 1536, [1, 2, 3, 4, 5, 8]), (1024, 3072, [1, 2, 3, 4, 5, 8]), (2048, 6144, [1, 2, 3, 4]), (2560, 9728, [1, 2]), (4096, 12288, [1, 2])])
def test_which_sublayers_fold(hidden, inner, rows):
    """As many squares as a block's threads ask for at their start, and the head's blocks, which have little else, only with a wide matrix and few rows."""
    from spyinfer_amd.parts.embedding import LMHead
    w_in, w_out = torch.zeros((2 * inner, hidden), device=DEV), torch.zeros((hidden, inner), device=DEV)
    assert [m for m in range(1, 10) if m != 6 and m != 7 and ops.folded_f32_pays(m, w_in, w_out)] == rows
    head = LMHead(4096, hidden)
    head.weight, head.weight_tiled = w_in, None

    class Batch:
        act_dtype = torch.float32

    fold = []
    for Batch.T in range(1, 10):
        if head.can_fold(Batch):
            fold.append(Batch.T)
    assert fold == {512: [], 1024: [], 2048: [1, 3, 4], 2560: [1], 4096: [1]}[hidden]


def test_caches_off_16_bytes_take_the_plain_kernels(tmp_path):
    """Decoding over caches that lie at 4 bytes: the same logits as over aligned ones, within rounding of float32 sums in another order."""
    from spyinfer_amd.engine.batch import StepEntry
    from spyinfer_amd.engine.runner import ModelRunner, load_model
    from spyinfer_amd.weights import write_random_model
    from tests.configs import INIT, TINY_D
    model = load_model(write_random_model(str(tmp_path / "m"), TINY_D, 64, torch.bfloat16, **INIT), "float32", DEV)
    prompts = [[5, 9, 200, 31], list(range(40, 77))]
    outs = []
    for shifted in (False, True):
        runner = ModelRunner(model, "float32", DEV, 16, 32, 2, enforce_eager=True, max_model_len=320)
        if shifted:
            for layer in runner.storage.layers.values():
                for name in ("k", "v"):
                    t = getattr(layer, name)
                    moved = torch.zeros(t.numel() + 1, device=DEV)[1:].view(t.shape)
                    assert moved.data_ptr() % 16 == 4
                    setattr(layer, name, moved)
        caches = [runner.manager.admit(i) for i in range(2)]
        for c, p in zip(caches, prompts):
            runner.manager.reserve(c, len(p))
        runner.step([StepEntry(c, p, []) for c, p in zip(caches, prompts)])
        got = []
        for t in (3, 250, 17):
            for c in caches:
                runner.manager.reserve(c, 1)
            got.append(runner.step([StepEntry(c, [t + i], [0]) for i, c in enumerate(caches)]).cpu().clone())
        outs.append(torch.stack(got))
    assert torch.allclose(outs[0], outs[1], rtol=2e-5, atol=2e-5), (outs[0] - outs[1]).abs().max()
