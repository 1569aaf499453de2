"""The gated delta rule over chunks of 16 tokens (csrc/delta_chunks.hip): entries of every length around a chunk and a few chunks, one
long enough for several segments, single tokens beside them, states carried from step to step, decays from none to all, one decay per
head and one per channel; against the recurrence in float64, token by token."""
import math

import pytest
import torch

from tests.gpu_util import require_gpu

pytestmark = pytest.mark.gpu


def walk(q, k, v, beta, decay, S):
    """One head: q, k, decay [T, d], v [T, dv], beta [T], S [d, dv] -> (o [T, dv], S)."""
    out = []
    for t in range(q.shape[0]):
        S = decay[t][:, None] * S
        u = beta[t] * (v[t] - S.T @ k[t])
        S = S + torch.outer(k[t], u)
        out.append(S.T @ q[t])
    return torch.stack(out), S


def unit(x):
    return x / torch.sqrt((x * x).sum(-1, keepdim=True) + 1e-6)


# heads, kv heads, key size, value size, decays per head (0: one per channel), lengths of the steps' entries
CASES = [(2, 1, 128, 128, 0, [(1, 17), (16, 31)]), (4, 2, 64, 48, 0, [(15, 1, 40), (2, 33, 1)]), (3, 3, 128, 16, 1, [(50, 5), (1, 1), (64, 2)]),
         (1, 1, 64, 32, 0, [(2300,), (7,)]), (2, 2, 128, 32, 1, [(1, 1, 1, 1, 2)]),
         # more blocks than compute units
         (11, 11, 128, 48, 0, [(17, 2, 16, 1, 33, 5, 1, 20), (1,) * 7 + (35,)])]


@pytest.mark.parametrize("how", ["slow", "fast", "mixed"])
@pytest.mark.parametrize("case", range(len(CASES)))
def test_chunks_against_the_recurrence(case, how):
    from spyinfer_amd.kernels import ops
    dev = require_gpu()
    H, G, d, dv, per_head, steps = CASES[case]
    if case == 3 and how != "slow":
        pytest.skip("the long entry once")
    dd = 1 if per_head else d
    g = torch.Generator().manual_seed(10 * case + len(how))
    slots, slot_ids = len(steps[0]) + 1, torch.randperm(len(steps[0]) + 1, generator=g)[:len(steps[0])].int()
    state = torch.randn(slots, H * d * dv + 8, generator=g) * 0.1
    S = [[state[int(s), h * d * dv:(h + 1) * d * dv].double().view(d, dv) for h in range(H)] for s in slot_ids]
    untouched = state[[i for i in range(slots) if i not in slot_ids.tolist()]].clone()
    state_dev = state.to(dev)
    a_log, dtb, nw = torch.rand(H, generator=g), torch.randn(H * dd, generator=g) * 0.1, 1.0 + 0.1 * torch.randn(dv, generator=g)
    for lens in steps:
        T = sum(lens)
        qkv = torch.randn(T, 2 * G * d + H * dv, generator=g)
        beta_pre = torch.randn(T, H, generator=g)
        # slow: decays near one; fast: most of the state is gone after a token; mixed: some channels of some tokens lose everything
        dec_pre = torch.randn(T, H * dd, generator=g) + {"slow": -6.0, "fast": 2.0, "mixed": -4.0}[how]
        if how == "mixed":
            dec_pre = torch.where(torch.rand(dec_pre.shape, generator=g) < 0.1, torch.full_like(dec_pre, 300.0), dec_pre)
        gate = torch.randn(T, H * dv, generator=g)
        cu = torch.tensor([0] + list(torch.tensor(lens).cumsum(0)), dtype=torch.int32)
        y = ops.delta_rule(qkv.to(dev), beta_pre.clone().to(dev), dec_pre.clone().to(dev), a_log.to(dev), dtb.to(dev), gate.to(dev), nw.to(dev), 1e-6,
                           state_dev, cu.to(dev), slot_ids.to(dev), H, G, d, dv).cpu().double().view(T, H, dv)
        x = qkv.double()
        q, k = unit(x[:, :G * d].view(T, G, d)) * d ** -0.5, unit(x[:, G * d:2 * G * d].view(T, G, d))
        v, beta = x[:, 2 * G * d:].view(T, H, dv), torch.sigmoid(beta_pre.double())
        dt = torch.nn.functional.softplus(dec_pre.double() + dtb.double()).view(T, H, dd).expand(T, H, d)
        decay = torch.exp(-torch.exp(a_log.double())[None, :, None] * dt)
        for e, n in enumerate(lens):
            at = slice(int(cu[e]), int(cu[e + 1]))
            for h in range(H):
                o, S[e][h] = walk(q[at, h // (H // G)], k[at, h // (H // G)], v[at, h], beta[at, h], decay[at, h], S[e][h])
                ref = o / torch.sqrt((o * o).mean(-1, keepdim=True) + 1e-6) * nw.double() * torch.sigmoid(gate[at].double().view(n, H, dv)[:, h])
                # float32 sums of up to 2 d terms of size one, over a root mean square: a few hundred roundings of 2^-24 of the largest
                assert float((y[at, h] - ref).abs().max()) < 2e-5 * max(1.0, float(ref.abs().max())), (e, h, n)
                got = state_dev[int(slot_ids[e]), h * d * dv:(h + 1) * d * dv].cpu().double().view(d, dv)
                assert float((got - S[e][h]).abs().max()) < 1e-5 * max(1.0, float(S[e][h].abs().max())), (e, h, n)
    assert torch.equal(state_dev.cpu()[[i for i in range(slots) if i not in slot_ids.tolist()]], untouched)


def test_an_infinite_value_stays_with_the_tokens_that_read_it():
    from spyinfer_amd.kernels import ops
    dev = require_gpu()
    g = torch.Generator().manual_seed(1)
    T, d, dv = 40, 64, 16
    qkv = torch.randn(T, 2 * d + dv, generator=g)
    qkv[21, 2 * d + 3] = float("inf")
    cu, slot = torch.tensor([0, T], dtype=torch.int32).to(dev), torch.zeros(1, dtype=torch.int32).to(dev)
    ones = lambda *s: torch.ones(*s, device=dev)
    y = ops.delta_rule(qkv.to(dev), ones(T, 1) * 0.3, ones(T, d) * -3, ones(1), ones(d), ones(T, dv), ones(dv), 1e-6, torch.zeros(1, d * dv, device=dev), cu, slot, 1, 1, d, dv)
    assert bool(y[:21].isfinite().all()) and not bool(y[21:].isfinite().all(dim=1).any())


# heads, key size, value size, lengths of the steps' entries
MEMORIES = [(2, 128, 128, [(1, 17), (16, 31)]), (3, 64, 48, [(15, 1, 40), (2, 33, 1)]), (1, 128, 16, [(150, 65), (1, 1), (64, 2)]), (1, 64, 32, [(2200,), (7,)])]


@pytest.mark.parametrize("how", ["keep", "lose", "wild"])
@pytest.mark.parametrize("case", range(len(MEMORIES)))
def test_matrix_memory_chunks_against_the_recurrence(case, how):
    """The mLSTM likewise; its gates: little forgotten, much forgotten, both with inputs that move the running maximum about."""
    from spyinfer_amd.kernels import ops
    dev = require_gpu()
    H, d, dv, steps = MEMORIES[case]
    if case == 3 and how != "keep":
        pytest.skip("the long entry once")
    g = torch.Generator().manual_seed(20 * case + len(how))
    n = len(steps[0])
    slot_ids = torch.randperm(n + 1, generator=g)[:n].int()
    state = torch.zeros(n + 1, ops.mlstm_state_size(H, d, dv))
    spare = [i for i in range(n + 1) if i not in slot_ids.tolist()]
    state[spare] = 7.0
    state_dev, cap = state.to(dev), 15.0
    S, N, M = ([[torch.zeros(z, dtype=torch.float64) for _ in range(H)] for _ in range(n)] for z in ((d, dv), (d,), ()))
    bi, bf, nw = torch.randn(H, generator=g), torch.randn(H, generator=g), 1.0 + 0.1 * torch.randn(H * dv, generator=g)
    for lens in steps:
        T = sum(lens)
        x = torch.randn(T, 2 * H * d + 2 * H * dv, generator=g)
        gates = torch.randn(T, 2 * H, generator=g) * {"keep": 0.5, "lose": 0.5, "wild": 9.0}[how]
        gates[:, H:] += {"keep": 4.0, "lose": -3.0, "wild": 0.0}[how]
        cu = torch.tensor([0] + list(torch.tensor(lens).cumsum(0)), dtype=torch.int32)
        y = ops.mlstm(x.to(dev), 0, H * d, 2 * H * d, 2 * H * d + H * dv, gates.clone().to(dev), bi.to(dev), bf.to(dev), cap, nw.to(dev), 1e-6, state_dev,
                      cu.to(dev), slot_ids.to(dev), H, d, dv).cpu().double().view(T, H, dv)
        xd = x.double()
        q, k = xd[:, :H * d].view(T, H, d) * d ** -0.5, xd[:, H * d:2 * H * d].view(T, H, d)
        v, og = xd[:, 2 * H * d:2 * H * d + H * dv].view(T, H, dv), torch.sigmoid(xd[:, 2 * H * d + H * dv:]).view(T, H, dv)
        ig = cap * torch.tanh((gates[:, :H].double() + bi.double()) / cap)
        fg = torch.nn.functional.logsigmoid(cap * torch.tanh((gates[:, H:].double() + bf.double()) / cap))
        for e, L in enumerate(lens):
            for h in range(H):
                for t in range(int(cu[e]), int(cu[e]) + L):
                    new = torch.maximum(fg[t, h] + M[e][h], ig[t, h])
                    a, b = torch.exp(fg[t, h] + M[e][h] - new), torch.exp(ig[t, h] - new)
                    S[e][h] = a * S[e][h] + b * torch.outer(k[t, h], v[t, h])
                    N[e][h] = a * N[e][h] + b * k[t, h]
                    M[e][h] = new
                    nq = float(N[e][h] @ q[t, h])
                    den = max(abs(nq), math.exp(-new)) + 1e-6
                    o = S[e][h].T @ q[t, h] / den
                    ref = o / torch.sqrt((o * o).mean() + 1e-6) * nw.double().view(H, dv)[h] * og[t, h]
                    # float32: a value of S^T q is rounded by at most 100 times 2^-24 of the sum of its terms' sizes (chains of 36 products,
                    # the parts' sums, the state's own roundings of the last chunks), and the head's norm divides by its root mean square
                    terms = float((S[e][h].abs().T @ q[t, h].abs()).max()) / den
                    bound = 100 * 2.0 ** -24 * terms / float(torch.sqrt((o * o).mean() + 1e-6)) * float((nw.double().view(H, dv)[h] * og[t, h]).abs().max())
                    assert float((y[t, h] - ref).abs().max()) < max(2e-5, bound), (e, h, t)
                st = state_dev[int(slot_ids[e])].cpu().double()
                head = st[h * (len(st) // H):(h + 1) * (len(st) // H)]
                assert float((head[:d * dv].view(d, dv) - S[e][h]).abs().max()) < 1e-5 * max(1.0, float(S[e][h].abs().max()))
                own = head[d * dv:].view(-1, d + 1)                          # n and m once for every slice of value channels
                assert float((own[:, :d] - N[e][h]).abs().max()) < 1e-5 * max(1.0, float(N[e][h].abs().max())) and float((own[:, d] - M[e][h]).abs().max()) < 1e-4
    assert bool((state_dev[spare] == 7.0).all())


@pytest.mark.parametrize("lengths", [[0, 20], [0, 0, 70, 0, 1]])
def test_entries_without_tokens_read_and_write_nothing(lengths):
    """The first entry's gates would lie before the rows; the other entries' results and states are those of a step without the empty ones."""
    from spyinfer_amd.kernels import ops
    dev = require_gpu()
    H, d, dv = 2, 64, 16
    g = torch.Generator().manual_seed(3)
    S, T = len(lengths), sum(lengths)
    state = torch.randn(S, ops.mlstm_state_size(H, d, dv), generator=g) * 0.1
    x, gates = torch.randn(T, 2 * H * d + 2 * H * dv, generator=g).to(dev), torch.randn(T, 2 * H, generator=g)
    bi, bf, nw = torch.randn(H, generator=g).to(dev), torch.randn(H, generator=g).to(dev), torch.ones(H * dv, device=dev)

    def run(entries):
        st = state.to(dev)
        cu = torch.tensor([0] + list(torch.tensor([lengths[e] for e in entries]).cumsum(0)), dtype=torch.int32).to(dev)
        y = ops.mlstm(x, 0, H * d, 2 * H * d, 2 * H * d + H * dv, gates.clone().to(dev), bi, bf, 15.0, nw, 1e-6, st, cu,
                      torch.tensor(entries, dtype=torch.int32).to(dev), H, d, dv)
        return y, st
    y, st = run(list(range(S)))
    y2, st2 = run([e for e in range(S) if lengths[e]])
    assert torch.equal(y, y2) and torch.equal(st, st2) and bool(y.isfinite().all())
    assert all(torch.equal(st[e].cpu(), state[e]) for e in range(S) if not lengths[e])


@pytest.mark.parametrize("d, dv", [(64, 16), (128, 256), (64, 24), (128, 8), (96, 64), (256, 64)])
def test_who_goes_by_chunks_is_known_to_the_plans(d, dv):
    import ctypes

    from spyinfer_amd.kernels import ops
    require_gpu()
    I = ctypes.c_int
    for f in (ops.hip().lib.spy_mlstm_workspace, ops.hip().lib.spy_delta_rule_workspace):
        assert (f(I(2), I(40), I(3), I(d), I(dv)) > 0) == ops.recurrence_by_chunks(d, dv) and f(I(5), I(5), I(3), I(d), I(dv)) == 0


@pytest.mark.parametrize("lengths", [[3, 1], [9, 1, 1], [40, 1], [17, 30, 2]])
def test_both_ways_give_the_same_results(lengths, monkeypatch):
    """Entries token by token where the longest is known to be short, by chunks where it is not known: the same read-outs and states
    to rounding, and the way that the caller's rule names."""
    from spyinfer_amd.kernels import ops
    dev = require_gpu()
    H, G, d, dv = 4, 2, 64, 32
    g = torch.Generator().manual_seed(8)
    S, T = len(lengths), sum(lengths)
    cu = torch.tensor([0] + list(torch.tensor(lengths).cumsum(0)), dtype=torch.int32).to(dev)
    sl = torch.arange(S, dtype=torch.int32).to(dev)
    rnd = lambda *s: torch.randn(*s, generator=g)
    qkv, beta, dec, gate, x, gates = rnd(T, 2 * G * d + H * dv), rnd(T, H), rnd(T, H * d) - 3, rnd(T, H * dv), rnd(T, 2 * H * d + 2 * H * dv), rnd(T, 2 * H)
    start = [rnd(S, H * d * dv) * 0.1, torch.zeros(S, ops.mlstm_state_size(H, d, dv))]
    ones = lambda n: torch.ones(n, device=dev)
    ways = []
    real = ops.hip().call
    monkeypatch.setattr(ops.hip(), "call", lambda name, *a: (ways.append(a[-2].value) if name in ("spy_delta_rule", "spy_mlstm") else None, real(name, *a))[1])
    out = []
    for longest in (None, max(lengths)):
        states = [s.to(dev) for s in start]
        y = [ops.delta_rule(qkv.to(dev), beta.to(dev), dec.to(dev), ones(H), ones(H * d), gate.to(dev), ones(dv), 1e-6, states[0], cu, sl, H, G, d, dv, longest=longest),
             ops.mlstm(x.to(dev), 0, H * d, 2 * H * d, 2 * H * d + H * dv, gates.clone().to(dev), ones(H), ones(H), 15.0, ones(H * dv), 1e-6, states[1], cu, sl, H, d, dv,
                       longest=longest)]
        out.append(y + states)
    assert ways == [1, 1] + [int(ops.recurrence_goes_by_chunks(S, T, H, d, dv, max(lengths), delta)) for delta in (True, False)]
    for a, b in zip(*out):
        # float32 sums of 64 products in other orders, over a root mean square: some dozens of roundings of 2^-24 of the largest
        assert float((a - b).abs().max()) < 1e-5 * max(1.0, float(b.abs().max()))
