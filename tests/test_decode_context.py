"""The position of a decoding step, without a GPU."""

import pytest
import torch

from petals_amd.ops.fused_decode import DecodeContext


@pytest.mark.parametrize("default", ["cpu", "meta"])
def test_position_with_another_default_device(default):
    """A process may have torch make its tensors elsewhere than where a session's position is."""
    ctx = DecodeContext(torch.device("cpu"))
    with torch.device(default):
        for p in (0, 7, 7900):
            ctx.set_position(p)
            assert (ctx.pos.tolist(), ctx.kv_len.tolist()) == ([p], [p + 1])
            ctx.advance()
            assert (ctx.pos.tolist(), ctx.kv_len.tolist()) == ([p + 1], [p + 2])
