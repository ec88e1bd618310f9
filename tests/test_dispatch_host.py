"""Which launches the modules choose, without a GPU: a stand-in for the library notes every call and refuses what the entry points refuse."""
import pytest
import torch

from fastfold_amd import _lib
from fastfold_amd.model.fastnn import _fused as F_

BF = torch.bfloat16


@pytest.fixture
def calls(monkeypatch):
    seen = []

    def call(name, *args):
        if name == "ffk_pair_bias" and args[7] not in (64, 128):
            raise RuntimeError("ffk_pair_bias: built for 64 or 128 pair channels, got %d" % args[7])
        seen.append(name)
    monkeypatch.setattr(_lib, "call", call)
    monkeypatch.setattr(_lib, "stream_ptr", lambda: 0)
    monkeypatch.setattr(F_, "check_cuda", lambda *ts: None)
    return seen


def _module(cls, *args, **kw):
    return cls(*args, **kw).to(BF).eval()


@pytest.mark.parametrize("r", [32, 64, 96, 128, 160])
@pytest.mark.parametrize("ending", [False, True])
def test_triangle_attention_of_256_channels_is_taken_at_every_length(calls, r, ending):
    """The kernel of short rows is built for 256 channels, the launch that makes its pair bias is not."""
    from fastfold_amd.model.fastnn import ops
    mod = _module(ops.ChunkTriangleAttentionEndingNode if ending else ops.ChunkTriangleAttentionStartingNode, 256, 0.25, c=32, n_head=8)
    with torch.no_grad():
        mod(torch.zeros(1, r, r, 256, dtype=BF), torch.ones(1, r, r, dtype=BF))
    assert "ffk_attention_fwd" in calls and "ffk_attention_block" not in calls
