"""Attention of entries with many rows and entries with few in one launch (csrc/attention_mixed.hip), against the plain formula in
float64 and against the two launches it stands for: every option, both head sizes and kinds of pages, one tile a block and two."""
import pytest
import torch

from tests.gpu_util import close, require_gpu
from tests.test_gpu_attention_f32 import plain
from tests.test_gpu_kernels import make_attention_case

pytestmark = pytest.mark.gpu

# n_q, n_kv, d, page, entries (cached, new), options
CASES = [
    (8, 2, 128, 16, [(0, 33), (40, 1), (0, 1)], {}),
    (8, 2, 64, 16, [(70, 1), (0, 129), (3, 2), (255, 1), (256, 1)], {}),
    (4, 4, 64, 64, [(0, 70), (300, 3), (63, 1), (64, 1)], {}),
    (4, 4, 128, 128, [(0, 5), (130, 66), (900, 1)], {}),
    (16, 8, 128, 8, [(0, 40), (517, 1), (0, 7)], {}),                       # eight waves, some without a block of keys
    (8, 2, 128, 16, [(200, 40), (300, 1), (90, 2)], dict(window=50)),
    (8, 2, 64, 16, [(200, 40), (300, 1), (90, 2)], dict(chunk=64)),
    (8, 2, 128, 16, [(0, 40), (77, 1)], dict(softcap=8.0)),
    (8, 2, 64, 16, [(0, 40), (77, 1)], dict(distance=True)),
    (8, 2, 128, 16, [(0, 40), (77, 1)], dict(sink=True)),
    (8, 2, 64, 32, [(0, 40), (77, 1)], dict(gate=True)),
    (128, 128, 64, 16, [(0, 300), (9, 1), (0, 3)], {}),                     # 384 pairs: two tiles a block
]


@pytest.mark.parametrize("case", range(len(CASES)))
def test_mixed_attention(case, monkeypatch):
    from spyinfer_amd.kernels import ops
    dev = require_gpu()
    n_q, n_kv, d, P, entries, opt = CASES[case]
    q, kc, vc, bt, te, ps, meta = make_attention_case(torch.bfloat16, dev, n_q, n_kv, d, P, entries, seed=300 + case, spike=True)
    g = torch.Generator().manual_seed(case)
    window, chunk, softcap = opt.get("window"), opt.get("chunk"), opt.get("softcap", 0.0)
    distance = torch.rand(2, n_q, generator=g) if opt.get("distance") else None
    sink = torch.randn(n_q, generator=g) if opt.get("sink") else None
    gate = torch.randn(q.shape, generator=g).to(torch.bfloat16) if opt.get("gate") else None
    on = lambda t: None if t is None else t.to(dev)
    launches = []
    call = ops.hip().call
    monkeypatch.setattr(ops.hip(), "call", lambda name, *a: (launches.append(name), call(name, *a))[1])
    def run():
        return ops.paged_attention(on(q), on(kc), on(vc), P, meta, n_q, n_kv, d, 0.11, window, softcap=softcap, distance=on(distance),
                                   sink=on(sink), chunk=chunk, gate=on(gate))
    got = run()
    assert launches == ["spy_attention_mixed"]
    ref = plain(q, kc, vc, P, bt, te, ps, n_q, n_kv, d, 0.11, window, chunk, softcap, distance, sink, gate)
    close(got, ref, torch.bfloat16, scale=3.0, what="mixed attention, case %d" % case)
    monkeypatch.setattr(ops, "mixed_attention_pays", lambda *a: False)
    apart = run()
    assert launches[1:] == ["spy_attention_prefill", "spy_attention_mfma"]
    close(got, apart, torch.bfloat16, scale=3.0, what="mixed attention against two launches, case %d" % case)
    if got.shape[0] <= ops.FUSED_DECODE_MAX_ROWS and ops.attention_hands_over_operand_rows(torch.bfloat16, n_q, d, P):
        monkeypatch.undo()
        rows = ops.paged_attention(on(q), on(kc), on(vc), P, meta, n_q, n_kv, d, 0.11, window, softcap=softcap, distance=on(distance), sink=on(sink),
                                   chunk=chunk, gate=on(gate), for_product=True)
        assert isinstance(rows, ops.OperandRows) and torch.equal(rows.to_rows(), got)
