"""Which steps' attention takes the raw product: what is asked, and in which order."""
import types

import pytest
import torch

from spyinfer_amd.kernels import ops


class Untouched:
    """A tensor's stand-in that nothing may be asked of."""

    def __getattr__(self, name):
        raise AssertionError("asked for %s" % name)


def _meta(S, T, longest):
    return types.SimpleNamespace(S=S, T=T, max_q_len=longest, tiles={"small": (None, None, T), "big": (None, None, 0)}, tiles_group=4)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_a_prompt_is_turned_away_before_any_tensor_is_asked(dtype):
    """The host asks once a layer, and bounds short prompts."""
    for meta in (_meta(1, 60, 60), _meta(3, 5, 3)):
        assert not ops.fused_attention_ok(dtype, meta, 16, 4, 128, 16, 128, Untouched(), Untouched(), (Untouched(), Untouched()))


def test_float32_operands_off_16_bytes():
    meta = _meta(2, 2, 1)
    on, off = torch.zeros(64), torch.zeros(65)[1:]
    assert on.data_ptr() % 16 == 0 and off.data_ptr() % 16 == 4
    ask = lambda dtype, *operands: ops.fused_attention_ok(dtype, meta, 16, 4, 128, 16, 128, None, None, operands)
    assert ask(torch.float32, on, on, None) and not ask(torch.float32, on, off) and not ask(torch.float32, off, on)
    assert ask(torch.bfloat16, off, off) == ask(torch.bfloat16)          # (bfloat16 rows: as it was, by the kernel's own check)
