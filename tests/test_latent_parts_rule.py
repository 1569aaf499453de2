"""Steps of single tokens through latent attention: how many shapes a growing request takes, each of which a graph is captured for."""
import types

import pytest
import torch

from spyinfer_amd.engine.runner import ModelRunner
from spyinfer_amd.kernels import ops
from spyinfer_amd.parts import LatentAttention, RotaryEmbedding


def shapes(heads, requests, window=None, longest=4096):
    """What the part's plan adds to the graph's key while ``requests`` requests grow to ``longest`` tokens."""
    part = LatentAttention(2048, heads, 128, 64, 128, 512, 0.07, 1e-6, RotaryEmbedding(64, 10000.0, 64), window=window)
    seen = set()
    for keys in range(1, longest + 1):
        batch = types.SimpleNamespace(T=requests, S=requests, max_q_len=1, max_kv_len=keys, act_dtype=torch.bfloat16, shared={}, keys={})
        batch.add_graph_key = batch.keys.__setitem__
        part.plan(batch)
        seen.add(tuple(batch.keys.items()))
    return len(seen)


@pytest.mark.parametrize("heads,window", [(16, None), (16, 1024), (32, None)])
def test_a_growing_request_takes_few_shapes(heads, window):
    counts = [shapes(heads, n, window) for n in range(1, 9)]
    assert max(counts) <= 7 and sum(counts) <= ModelRunner.MAX_GRAPHS // 4


def test_parts_fit_the_kernel_and_the_chip():
    for tiles in (1, 2, 5, 12, 31, 64, 255, 256):
        most = min(32, 256 // tiles)
        for keys in range(1, 3000, 7):
            parts, chunks = ops.latent_few_key_parts(tiles, keys), -(-keys // 32)
            assert 1 <= parts <= most and parts >= min(chunks, most)
            assert parts < 2 * chunks
