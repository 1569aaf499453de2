"""Attention of entries with many rows whose 128-row tiles are few: one tile a block where every block has a compute unit,
two where not, the keys in parts or not by what the entries with such tiles read, beside single tokens with more keys."""
import pytest
import torch

from tests.gpu_util import close, require_gpu
from tests.test_gpu_kernels import make_attention_case, plain_paged_attention

# n_q, n_kv, d, page, entries (cached, new), window, parts expected
CASES = [
    (8, 2, 128, 16, [(0, 33)], None, 1),                              # two tiles, the second with four rows
    (8, 8, 64, 16, [(0, 129), (5, 64)], None, 1),
    (4, 1, 128, 16, [(700, 40), (3, 1), (0, 200)], None, 2),           # parts: few tiles behind many keys
    (4, 1, 64, 16, [(900, 33), (2500, 1)], None, 3),                   # the same beside a single token with more keys
    (4, 1, 128, 16, [(0, 100), (1500, 1)], None, 1),                   # the single token's keys split nothing
    (4, 1, 64, 64, [(1500, 40)], 90, 1),                               # a window leaves nothing to split
    (256, 256, 64, 16, [(0, 130)], None, 1),                           # 512 pairs: two tiles a block
    (256, 128, 64, 16, [(0, 70)], None, 1),                            # 256 pairs: the most with one tile a block
]


@pytest.mark.gpu
@pytest.mark.parametrize("case", range(len(CASES)))
def test_few_tiles(case, monkeypatch):
    from spyinfer_amd.kernels import ops
    dev = require_gpu()
    n_q, n_kv, d, P, entries, window, parts = CASES[case]
    q, kc, vc, bt, te, ps, meta = make_attention_case(torch.bfloat16, dev, n_q, n_kv, d, P, entries, seed=90 + case, window=window, spike=True)
    group = n_q // n_kv
    meta.max_big_keys = max(a + n for a, n in entries if n * group >= 64)
    blocks = meta.tiles["big"][2] * n_kv
    assert blocks > 0
    keys = meta.max_big_keys if window is None else min(meta.max_big_keys, window + 128 // group + 1)
    assert ops.prefill_key_parts(blocks, keys, d) == parts
    ref = plain_paged_attention(q, kc, vc, P, bt, te, ps, n_q, n_kv, d, 0.11, window)
    # entries of both kinds: two launches, so that the large tiles' own launch is what is tested
    monkeypatch.setattr(ops, "mixed_attention_pays", lambda *a: False)
    launches = []
    real = ops.hip().call
    monkeypatch.setattr(ops.hip(), "call", lambda name, *a: (launches.append((name, a[23].value if name == "spy_attention_prefill" else None)), real(name, *a))[1])
    got = ops.paged_attention(q.to(dev), kc.to(dev), vc.to(dev), P, meta, n_q, n_kv, d, 0.11, window)
    assert launches[0] == ("spy_attention_prefill", parts) and [n for n, _ in launches[1:]] == ["spy_attention_mfma"] * (meta.tiles["small"][2] > 0)
    close(got, ref, torch.bfloat16, scale=3.0, what="few tiles, case %d" % case)


@pytest.mark.parametrize("blocks", [1, 8, 31, 104, 200, 255, 256, 4000])
def test_parts_stay_within_what_the_kernels_take(blocks):
    from spyinfer_amd.kernels import ops
    for keys in (1, 63, 64, 255, 256, 513, 2048, 40000):
        parts = ops.prefill_key_parts(blocks, keys)
        assert 1 <= parts <= 16 and (parts == 1 or (parts * blocks <= 512 and parts * 256 <= keys and blocks < 256))
