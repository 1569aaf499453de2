"""The fused attention of few single tokens in blocks of eight waves (csrc/attention_mfma.hip): contexts at the edges of a wave's, a part's and a page's
keys, the first token of a request, several parts and one, and steps on both sides of the line to blocks of four; against float64."""
import math

import numpy as np
import pytest
import torch

from tests.gpu_util import close, require_gpu
from tests.test_gpu_kernels import _with_pieces, make_attention_case, plain_paged_attention, plain_qk, rnd

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("P,window", [(16, None), (64, None), (16, 300)])
@pytest.mark.parametrize("cached", [[0], [1, 31, 32, 33], [255, 256, 257, 0, 511, 512, 513, 1023], [2100, 4], [5] * 21, [40 + 61 * i for i in range(20)]])
def test_few_single_tokens(cached, P, window):
    from spyinfer_amd.kernels import key_pieces, ops
    from spyinfer_amd.parts.rotary import RotaryEmbedding
    dev = require_gpu()
    n_q, n_kv, d, dtype, eps, theta = 16, 8, 128, torch.bfloat16, 1e-6, 1e6
    assert key_pieces.piece_waves(len(cached), n_kv, d) == (8 if len(cached) <= 20 else 4)
    _q, kc, vc, bt, te, ps, meta = make_attention_case(dtype, dev, n_q, n_kv, d, P, [(a, 1) for a in cached], seed=len(cached), window=window)
    rec = _with_pieces(meta, [a + 1 for a in cached], n_kv, window, d, dev)
    assert window or max(cached) < 400 or rec[:, 5].max() > 1
    T = len(cached)
    qkv = rnd((T, (n_q + 2 * n_kv) * d), dtype, "cpu", 7)
    qw, kw = ((1 + 0.2 * rnd((d,), torch.float32, "cpu", s)).to(dtype) for s in (8, 9))
    pos = torch.tensor(cached, dtype=torch.int32)
    rope = RotaryEmbedding(d, theta, d)
    rope.prepare(dev, 2200)
    rq, rk, rv = plain_qk(qkv, n_q, n_kv, d, qw, kw, eps, theta, d, pos)
    kc_ref, vc_ref = kc.clone(), vc.clone()
    for s, a in enumerate(cached):
        page = bt[s][a // P]
        kc_ref[page, :, a % P, :] = rk[s].to(dtype)
        vc_ref[page, :, :, a % P] = rv[s].to(dtype)
        kc[page, :, a % P, :] = float("nan")                          # (read before it is written, it would show)
        vc[page, :, :, a % P] = float("nan")
    ref = plain_paged_attention(rq.reshape(T, n_q * d).to(dtype), kc_ref, vc_ref, P, bt, te, ps, n_q, n_kv, d, d ** -0.5, window)
    kd, vd = kc.to(dev), vc.to(dev)
    raw = ops.RawQKV(qkv.to(dev), qw.to(dev), kw.to(dev), eps, rope.cos, rope.sin, True)
    out = ops.paged_attention(None, kd, vd, P, meta, n_q, n_kv, d, d ** -0.5, window, raw)
    close(out, ref, dtype, scale=3.0, what="attention of few tokens")
    same = lambda a, b: torch.equal(torch.nan_to_num(a.float().cpu(), nan=-77.0), torch.nan_to_num(b.float(), nan=-77.0))
    assert same(vd, vc_ref), "values must be stored unchanged, and nothing else written"
    # a second call on what the first one stored: the counters are as they were
    again = ops.paged_attention(None, kc_ref.to(dev), vc_ref.to(dev), P, meta, n_q, n_kv, d, d ** -0.5, window, raw)
    assert torch.equal(again, out)
    raw.store = False                                                   # (the new key read from the cache, where another call put it)
    close(ops.paged_attention(None, kd, vd, P, meta, n_q, n_kv, d, d ** -0.5, window, raw), ref, dtype, scale=3.0, what="without store")


def test_steps_whose_longest_request_passes_the_line(tmp_path):
    """18 requests of 8 kv heads, the longest passing 1024 keys while they decode under graphs: blocks of eight waves, then of four, which are two graphs; the
    same logits as eager steps, and the graphs go by the longest request."""
    from spyinfer_amd.engine.batch import StepEntry
    from spyinfer_amd.engine.runner import ModelRunner, load_model
    from spyinfer_amd.weights import write_random_model
    from tests.configs import INIT, TINY_E
    require_gpu()
    config = dict(TINY_E, num_hidden_layers=1, num_key_value_heads=8, max_position_embeddings=1100)
    model = load_model(write_random_model(str(tmp_path / "m"), config, 5, torch.bfloat16, **INIT), "bfloat16", "cuda:0")
    gen = torch.Generator().manual_seed(9)
    prompts = [torch.randint(0, 300, (1020 if i == 3 else 30 + 7 * i,), generator=gen).tolist() for i in range(18)]
    runs = []
    for eager in (True, False):
        runner = ModelRunner(model, "bfloat16", "cuda:0", 16, 300, 18, enforce_eager=eager, max_model_len=1100)
        caches = [runner.manager.admit(i) for i in range(18)]
        for c, p in zip(caches, prompts):
            runner.manager.reserve(c, len(p))
        runner.step([StepEntry(c, p, []) for c, p in zip(caches, prompts)])
        outs, tokens = [], torch.Generator().manual_seed(10)
        for _ in range(9):
            step = torch.randint(0, 300, (18,), generator=tokens).tolist()
            for c in caches:
                runner.manager.reserve(c, 1)
            outs.append(runner.step([StepEntry(c, [t], [0]) for c, t in zip(caches, step)]).cpu().clone())
        runs.append(outs)
    assert sorted(dict(key[2])["decode_pieces_waves_8_0_128"] for key in runner._graphs) == [4, 8]
    assert runner.graph_replays == 7                                    # (of 4 steps and 5, the first of each shape runs kernel by kernel)
    assert all(torch.equal(a, b) for a, b in zip(*runs)) and all(torch.isfinite(a).all() for a in runs[0])
