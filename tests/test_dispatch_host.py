"""Which launches the modules choose, without a GPU: a stand-in for the library notes every call and refuses what the entry points refuse."""
import pytest
import torch

from fastfold_amd import _lib
from fastfold_amd.model.fastnn import _fused as F_
from fastfold_amd.model.fastnn.kernel import LayerNorm

BF = torch.bfloat16


@pytest.fixture
def calls(monkeypatch):
    seen = []

    def call(name, *args):
        if name == "ffk_pair_bias" and args[7] not in (64, 128):
            raise RuntimeError("ffk_pair_bias: built for 64 or 128 pair channels, got %d" % args[7])
        at = {"ffk_attention_block": (3, 4), "ffk_attention_heads": (2, 3), "ffk_transition_block": (3, 4, 8)}.get(name, ())
        if any(args[i] % 16 for i in at):                     # gamma, beta (and the transition's second bias)
            raise RuntimeError("%s: buffers must be 16-byte aligned" % name)
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


def _modules():
    from fastfold_amd.model.fastnn import msa, ops

    def pair(r, c):
        return torch.zeros(1, r, r, c, dtype=BF), torch.ones(1, r, r, dtype=BF)

    def seqs(s, r, c):
        return torch.zeros(1, s, r, c, dtype=BF), torch.ones(1, s, r, dtype=BF)
    yield ops.ChunkTriangleAttentionStartingNode(128, 0.25, c=32, n_head=4), pair(64, 128)
    yield ops.ChunkTriangleAttentionEndingNode(64, 0.25, c=16, n_head=4), pair(96, 64)
    for r in (96, 160):
        m, mask = seqs(128, r, 256)
        yield msa.MSARowAttentionWithPairBias(256, 128, c=32, n_head=8), (m, pair(r, 128)[0], mask)
    m, mask = seqs(128, 96, 64)
    yield msa.MSARowAttentionWithPairBias(64, 128, c=8, n_head=8), (m, pair(96, 128)[0], mask)
    yield msa.MSAColumnAttention(256), seqs(128, 96, 256)
    yield ops.Transition(64), (torch.zeros(1, 40, 96, 64, dtype=BF),)


@pytest.mark.parametrize("i", range(7))
def test_normalisation_weights_may_lie_anywhere(calls, i):
    """Parameters that are slices of one flat buffer need not begin on 16 bytes: the launches that read them element by element take
    them, as they take every other module whose kernel wants them aligned."""
    mod, args = list(_modules())[i]
    mod = mod.to(BF).eval()
    for aligned in (True, False):
        del calls[:]
        for m in mod.modules():
            if isinstance(m, LayerNorm) and not aligned:
                for p in (m.weight, m.bias):
                    p.data = torch.ones(p.numel() + 8, dtype=BF)[1:p.numel() + 1]
        with torch.no_grad():
            mod(*args)
        short = [n for n in calls if n in ("ffk_attention_block", "ffk_attention_heads", "ffk_transition_block")]
        assert bool(short) == aligned, calls


@pytest.mark.parametrize("r", [32, 96, 128, 160, 224, 256, 384])
def test_the_route_of_an_attention_does_not_depend_on_the_number_of_rows(calls, r):
    """A share of the batch rows (a rank's, a caller's piece) gets the bits of the full call, so it takes the same launches."""
    from fastfold_amd.model.fastnn import msa
    row, ext, col = (_module(*a, **kw) for a, kw in (((msa.MSARowAttentionWithPairBias, 256, 128), dict(c=32, n_head=8)),
                                                     ((msa.MSARowAttentionWithPairBias, 64, 128), dict(c=8, n_head=8)),
                                                     ((msa.MSAColumnAttention, 256), {})))
    z = torch.zeros(1, r, r, 128, dtype=BF)
    for mod, c in ((row, 256), (ext, 64), (col, 256)):
        routes = set()
        for b2 in (1, 31, 33, 60, 130, 300):
            m = torch.zeros(1, r, b2, c, dtype=BF) if mod is col else torch.zeros(1, b2, r, c, dtype=BF)
            mask = torch.ones(m.shape[:3], dtype=BF)
            del calls[:]
            with torch.no_grad():
                mod(m, mask) if mod is col else mod(m, z, mask)
            routes.add(tuple(calls))
        assert len(routes) == 1, routes
