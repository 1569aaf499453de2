"""The float32 attention on the matrix cores (csrc/attention_f32.hip): every option of the attention, single tokens, portions and
mixes, one part of the keys and several, against the plain formula in float64; unused slots and given-back pages hold NaN."""
import math

import pytest
import torch

from tests.gpu_util import require_gpu
from tests.test_gpu_kernels import make_attention_case

pytestmark = pytest.mark.gpu


def plain(q, kc, vc, P, bt, token_entry, positions, n_q, n_kv, d, scale, window=None, chunk=None, softcap=0.0, distance=None, sink=None, gate=None):
    T = q.shape[0]
    out = torch.zeros(T, n_q, d, dtype=torch.float64)
    for t in range(T):
        s, p = int(token_entry[t]), int(positions[t])
        lo = p - p % chunk if chunk else (max(0, p - window + 1) if window else 0)
        keys = range(lo, p + 1)
        K = torch.stack([kc[bt[s][c // P], :, c % P, :] for c in keys]).double().repeat_interleave(n_q // n_kv, dim=1)
        V = torch.stack([vc[bt[s][c // P], :, :, c % P] for c in keys]).double().repeat_interleave(n_q // n_kv, dim=1)
        x = torch.einsum("khd,hd->hk", K, q[t].double().view(n_q, d)) * scale
        if softcap:
            x = softcap * torch.tanh(x / softcap)
        if distance is not None:
            x = x - distance[0].double()[:, None] * torch.log1p(distance[1].double()[:, None] * (p - torch.tensor(list(keys))).double()[None])
        if sink is not None:
            x = torch.cat([x, sink.double()[:, None]], dim=1)
        out[t] = torch.einsum("hk,khd->hd", torch.softmax(x, dim=1)[:, :len(keys)], V)
    out = out.view(T, n_q * d)
    return out if gate is None else out * torch.sigmoid(gate.double())


# n_q, n_kv, d, page, entries (cached, new), options
CASES = [
    (16, 8, 128, 16, [(0, 37)], {}),
    (4, 2, 64, 16, [(0, 1)], {}),
    (4, 4, 64, 48, [(15, 1), (16, 1), (17, 1), (0, 3)], {}),
    (16, 8, 128, 16, [(900, 1), (31, 1), (0, 1), (415, 1)], {}),               # single tokens, keys in several parts
    (6, 2, 128, 32, [(500, 30), (0, 70), (129, 1)], dict(window=100)),
    (6, 2, 64, 16, [(300, 1), (40, 2)], dict(window=16)),
    (8, 8, 128, 16, [(250, 20), (47, 1)], dict(chunk=48)),
    (4, 1, 128, 64, [(700, 5)], dict(chunk=100, sink=True)),
    (5, 1, 64, 16, [(100, 9), (600, 1)], dict(softcap=3.0, distance=True, sink=True, gate=True)),
    (16, 2, 128, 16, [(70, 40)], dict(distance=True, gate=True)),
    (32, 1, 64, 16, [(33, 3)], dict(softcap=2.0)),                             # a group of more heads than a tile has rows
]


@pytest.mark.parametrize("case", range(len(CASES)))
def test_float32_attention(case, monkeypatch):
    from spyinfer_amd.kernels import ops
    dev = require_gpu()
    n_q, n_kv, d, P, entries, options = CASES[case]
    opt = dict(options)
    q, kc, vc, bt, te, ps, meta = make_attention_case(torch.float32, dev, n_q, n_kv, d, P, entries, seed=100 + case, spike=True)
    g = torch.Generator().manual_seed(case)
    T = q.shape[0]
    if opt.pop("sink", None):
        opt["sink"] = torch.randn(n_q, generator=g)
    if opt.pop("distance", None):
        opt["distance"] = torch.rand(2, n_q, generator=g)
    wide = None
    if opt.pop("gate", None):
        wide = torch.randn(T, n_q * d + 12, generator=g)                       # the gate's rows lie in a wider product
        opt["gate"] = wide[:, 4:4 + n_q * d]
    scale = 1.0 / math.sqrt(d)
    ref = plain(q, kc, vc, P, bt, te, ps, n_q, n_kv, d, scale, **opt)
    reach = opt.get("window") or opt.get("chunk")
    if reach:                                                                  # pages that no query reads any more are gone
        table = torch.tensor(bt, dtype=torch.int32)
        for s, (a, _) in enumerate(entries):
            lo = a - a % reach if "chunk" in opt else max(0, a - reach + 1)
            table[s, :lo // P] = -1
        meta.block_table = table.to(dev)
    G = n_q // n_kv
    rows = [(s, r0) for s, (_, n) in enumerate(entries) for r0 in range(0, n * G, 16)]
    i32 = lambda x: torch.tensor(x, dtype=torch.int32, device=dev)
    meta.tiles = {"small": (i32([s for s, _ in rows]), i32([r for _, r in rows]), len(rows)), "big": (i32([]), i32([]), 0)}
    called = []
    real = ops.hip().call
    monkeypatch.setattr(ops.hip(), "call", lambda name, *a: (called.append(name), real(name, *a))[1])
    on = {k: (v.to(dev) if torch.is_tensor(v) else v) for k, v in opt.items() if k != "gate"}
    if wide is not None:
        on["gate"] = wide.to(dev)[:, 4:4 + n_q * d]
    out = ops.paged_attention(q.to(dev), kc.to(dev), vc.to(dev), P, meta, n_q, n_kv, d, scale, on.pop("window", None), **on).cpu().double()
    assert called == ["spy_attention_f32"]
    # scores up to 100 here: each is rounded by d / 2 products or so, which moves a weight by that much relatively: 2e-5 of the largest value
    assert float((out - ref).abs().max()) < 2e-5 * max(1.0, float(vc[~vc.isnan()].abs().max()))


# n_q, n_kv, d, page, entries (cached, new), options, (entry, position, kv head, dim, value) of what is not finite
HIDDEN = [
    (4, 2, 64, 16, [(0, 21)], {}, [(0, 9, 0, 3, "inf"), (0, 17, 1, 63, "nan")]),                    # a later token of the portion
    (8, 8, 128, 16, [(300, 20), (5, 2)], {}, [(0, 311, 2, 100, "-inf"), (1, 6, 7, 0, "nan")]),       # the same behind keys in parts
    (8, 2, 128, 32, [(70, 3)], dict(window=40), [(0, 31, 1, 5, "nan"), (0, 32, 0, 77, "inf")]),      # just before a window, in its first block
    (8, 2, 64, 16, [(88, 1), (86, 12)], dict(chunk=41), [(0, 81, 0, 1, "inf"), (1, 80, 1, 2, "nan")]),
    (8, 1, 128, 16, [(0, 18)], dict(window=5), [(0, 15, 0, 9, "inf"), (0, 15, 0, 10, "-inf"), (0, 16, 0, 9, "inf")]),
]


@pytest.mark.parametrize("case", range(len(HIDDEN)))
def test_a_value_that_is_not_finite_stays_with_the_rows_that_read_it(case):
    """Rows of one 16-row tile read different keys; a weight of zero would not take an infinity or a NaN away."""
    from spyinfer_amd.kernels import ops
    dev = require_gpu()
    n_q, n_kv, d, P, entries, opt, odd = HIDDEN[case]
    q, kc, vc, bt, te, ps, meta = make_attention_case(torch.float32, dev, n_q, n_kv, d, P, entries, seed=130 + case)
    for s, c, hk, j, x in odd:
        vc[bt[s][c // P], hk, j, c % P] = float(x)
    G = n_q // n_kv
    rows = [(s, r0) for s, (_, n) in enumerate(entries) for r0 in range(0, n * G, 16)]
    i32 = lambda x: torch.tensor(x, dtype=torch.int32, device=dev)
    meta.tiles = {"small": (i32([s for s, _ in rows]), i32([r for _, r in rows]), len(rows)), "big": (i32([]), i32([]), 0)}
    ref = plain(q, kc, vc, P, bt, te, ps, n_q, n_kv, d, d ** -0.5, **opt)
    on = dict(opt)
    out = ops.paged_attention(q.to(dev), kc.to(dev), vc.to(dev), P, meta, n_q, n_kv, d, d ** -0.5, on.pop("window", None), **on).cpu().double()
    fine = ref.isfinite()
    assert bool(fine.any()) and (case == 3 or not bool(fine.all()))
    assert bool(out[fine].isfinite().all())
    assert float((out - ref)[fine].abs().max()) < 2e-5 * float(vc[vc.isfinite()].abs().max())      # (as above)
    assert torch.equal(torch.nan_to_num(out[~fine], nan=7.0), torch.nan_to_num(ref[~fine], nan=7.0))


# entries (cached, new), window, chunk, parts of the keys
PARTS = [([(0, 5)], None, None, 1), ([(100, 28)], None, None, 1), ([(100, 29)], None, None, 2), ([(15, 1)], None, None, 2), ([(600, 1)], None, None, 6),
         ([(600, 1)], 16, None, 1), ([(600, 1)], 112, None, 1), ([(600, 1)], 113, None, 2), ([(600, 1)], 300, None, 4), ([(600, 3)], None, 128, 1),
         ([(600, 3)], None, 129, 2), ([(700, 1)] * 40, None, None, 3)]


@pytest.mark.parametrize("case", range(len(PARTS)))
def test_parts_follow_the_keys_that_can_be_read(case, monkeypatch):
    """A window or chunk of a long context leaves little to split, and a short prompt nothing."""
    from spyinfer_amd.kernels import ops
    dev = require_gpu()
    entries, window, chunk, parts = PARTS[case]
    n_q, n_kv, d, P = 2, 2, 64, 16
    q, kc, vc, bt, te, ps, meta = make_attention_case(torch.float32, dev, n_q, n_kv, d, P, entries, seed=160 + case)
    rows = [(s, r0) for s, (_, n) in enumerate(entries) for r0 in range(0, n, 16)]
    i32 = lambda x: torch.tensor(x, dtype=torch.int32, device=dev)
    meta.tiles = {"small": (i32([s for s, _ in rows]), i32([r for _, r in rows]), len(rows)), "big": (i32([]), i32([]), 0)}
    seen = []
    real = ops.hip().call
    monkeypatch.setattr(ops.hip(), "call", lambda name, *a: (seen.append((name, a[22].value)), real(name, *a))[1])
    out = ops.paged_attention(q.to(dev), kc.to(dev), vc.to(dev), P, meta, n_q, n_kv, d, d ** -0.5, window, chunk=chunk).cpu().double()
    assert seen == [("spy_attention_f32", parts)]
    ref = plain(q, kc, vc, P, bt, te, ps, n_q, n_kv, d, d ** -0.5, window, chunk)
    assert float((out - ref).abs().max()) < 2e-5 * float(vc[vc.isfinite()].abs().max())
