"""ffk_transition_block (both layers of a transition in one kernel, weights in fragment order) through the C ABI against float64
(fastfold/model/fastnn/ops.py:71-82)."""
import pytest
import torch

pytestmark = pytest.mark.gpu
BF = torch.bfloat16
# Three roundings to bf16 behind the rounded rows (hidden value, update, and the float64 side's none): each by at most 2^-9 of a value.
TOL = 3 * 2.0 ** -9


# the edges of a workgroup's rows (64 or 128), of its 32-row tiles, and the row counts at which the layout changes
@pytest.mark.parametrize("C,factor,M", [(C, 4, M) for C in (64, 128, 256) for M in (1, 31, 64, 65, 127, 129, 1000)]
                         + [(64, 2, M) for M in (1, 33, 128, 129, 777)] + [(128, 4, 16384 + 33), (256, 4, 16384 + 33)])
@pytest.mark.parametrize("tail", [False, True])
def test_transition_block_against_float64(dev, C, factor, M, tail):
    from fastfold_amd import _lib
    from fastfold_amd.model.fastnn import _fused as F_
    g = torch.Generator().manual_seed(C + M)
    H = factor * C

    def rnd(*shape, scale=1.0, shift=0.0):
        return (torch.randn(*shape, generator=g) * scale + shift).to(dev, BF)
    x = rnd(M, C, scale=1.5, shift=0.3)
    gam, bet, b1, b2 = rnd(C, scale=0.1, shift=1.0), rnd(C, scale=0.1), rnd(H), rnd(C)
    w1, w2 = rnd(H, C, scale=C ** -0.5), rnd(C, H, scale=H ** -0.5)
    p1, p2 = F_.pack_transition_block(w1, w2, BF, dev)
    out, t = (x.clone() if tail else torch.empty_like(x)), (torch.zeros(M, C, dtype=torch.int8, device=dev) if tail else None)
    _lib.transition_block(out, out if tail else x, gam, bet, p1, b1, p2, b2, M=M, C=C, hidden=H, xtail=t)
    torch.cuda.synchronize()
    d = lambda v: v.double().cpu()                            # noqa: E731
    xd = d(x)
    mu = xd.mean(-1, keepdim=True)
    y = ((xd - mu) / torch.sqrt(((xd - mu) ** 2).mean(-1, keepdim=True) + 1e-5) * d(gam) + d(bet)).to(BF).double()
    upd = torch.relu(y @ d(w1).t() + d(b1)) @ d(w2).t() + d(b2)
    if tail:      # the result at 24 bits: its rounding to bf16 would be one of the stream, not of the update
        got = ((out.view(torch.int16).to(torch.int32) << 16) + (t.to(torch.int32) << 8)).view(torch.float32).double().cpu()
        assert float((got - xd - upd).norm() / upd.norm()) < TOL
    else:         # ... which is another 2^-9 of the result here
        assert float((d(out) - xd - upd).norm()) < TOL * float(upd.norm()) + 2.0 ** -9 * float((xd + upd).norm())


def test_transition_block_refuses(dev):
    from fastfold_amd import _lib
    x, v = torch.zeros(64, 96, dtype=BF, device=dev), torch.zeros(384, dtype=BF, device=dev)
    with pytest.raises(RuntimeError, match="built for"):
        _lib.transition_block(x, x, v, v, x, v, x, v, M=64, C=96, hidden=384)
    with pytest.raises(RuntimeError, match="built for"):
        _lib.transition_block(x, x, v, v, x, v, x, v, M=64, C=128, hidden=256)
    with pytest.raises(RuntimeError, match="bf16"):
        _lib.transition_block(x.float(), x.float(), v, v, x, v, x, v, M=64, C=64, hidden=256)


@pytest.mark.parametrize("C,M", [(C, M) for C in (128, 256) for M in (1, 63, 1000, 16384 - 40, 16384 + 40, 40000)])
@pytest.mark.parametrize("tail", [False, True])
def test_both_kernels_of_a_transition_give_the_same_bits(dev, C, M, tail):
    """Rows go to one or the other by their number, and a piece of the rows has to get the bits of all of them."""
    from fastfold_amd import _lib
    from fastfold_amd.model.fastnn import _fused as F_
    g = torch.Generator().manual_seed(C + M)
    H = 4 * C

    def rnd(*shape, scale=1.0, shift=0.0):
        return (torch.randn(*shape, generator=g) * scale + shift).to(dev, BF)
    x = rnd(M, C, scale=1.5, shift=0.3)
    gam, bet, b1, b2 = rnd(C, scale=0.1, shift=1.0), rnd(C, scale=0.1), rnd(H), rnd(C)
    w1, w2 = rnd(H, C, scale=C ** -0.5), rnd(C, H, scale=H ** -0.5)
    p1, p2 = F_.pack_transition_block(w1, w2, BF, dev)
    tails = [torch.randint(-100, 100, (M, C), generator=g, dtype=torch.int8).to(dev)] * 2 if tail else [None, None]
    tails = [t if t is None else t.clone() for t in tails]
    outs = [torch.empty_like(x), torch.empty_like(x)]
    _lib.transition_fused(outs[0], x, gam, bet, w1, b1, w2, b2, M=M, C=C, hidden=H, xtail=tails[0])
    _lib.transition_block(outs[1], x, gam, bet, p1, b1, p2, b2, M=M, C=C, hidden=H, xtail=tails[1])
    torch.cuda.synchronize()
    assert torch.equal(outs[0], outs[1]) and (not tail or torch.equal(tails[0], tails[1]))
