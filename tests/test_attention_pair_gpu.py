"""The bf16 attention core for heads of 32 channels with a bias and more than 256 keys (two batch rows and 32 queries per wave,
reference zero until a sum leaves its range) against float64: edges of its tiles, rows and workgroups, scores far from zero, rows
without keys."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu
BF = torch.bfloat16


def _case(dev, B2, H, N, shift, mask, v_scale=1.0):
    from fastfold_amd import _lib
    from fastfold_amd.model.fastnn.kernel import layouts
    g = torch.Generator().manual_seed(N * 7 + B2)
    q, k, v = (torch.randn(B2, H, N, 32, generator=g).to(BF) for _ in range(3))
    q, v = (q.float() * 0.25).to(BF), (v.float() * v_scale).to(BF)
    bias = torch.randn(H, N, N, generator=g) * 2
    if shift is not None:                       # log2 units added to every score of a query: nothing changes
        bias = bias + torch.tensor(shift).repeat(N // len(shift) + 1)[:N][None, :, None]
    bias = bias.to(BF)
    NT = layouts.n_tiles(N)
    kb, fl = torch.empty(B2, NT * 32, device=dev), torch.empty(B2, NT, dtype=torch.int32, device=dev)
    m = mask.to(dev, BF) if mask is not None else None
    _lib.key_bias(kb, fl, m, B=B2, N=N, **({} if m is None else dict(mask_sb=N, mask_sn=1)))
    out = torch.empty(B2, N, H * 32, dtype=BF, device=dev)
    d = lambda t: t.to(dev)
    _lib.attention_fwd(out, layouts.tile_qk(d(q)), layouts.tile_qk(d(k)), layouts.tile_v(d(v)), layouts.tile_bias(d(bias)), kb, fl, None,
                       B2=B2, H=H, Nq=N, Nk=N)
    torch.cuda.synchronize()
    s = q.double() @ k.double().transpose(-1, -2) + bias.double()
    if mask is not None:
        s = s.masked_fill(mask[:, None, None, :] == 0, -np.inf)
    top = s.max(-1, keepdim=True).values
    p = torch.exp2(s - torch.where(top.isfinite(), top, torch.zeros_like(top)))
    l = p.sum(-1, keepdim=True)
    want = torch.where(l > 0, (p @ v.double()) / l.clamp_min(1e-300), torch.zeros(()).double()).permute(0, 2, 1, 3).reshape(B2, N, H * 32)
    # probabilities rounded to bf16, in the numerator and in the denominator, and the result: at most 2^-8 each of the mean of |v|
    size = torch.where(l > 0, (p @ v.double().abs()) / l.clamp_min(1e-300), torch.zeros(()).double()).permute(0, 2, 1, 3).reshape(B2, N, H * 32)
    err = (out.cpu().double() - want).abs()
    assert bool((err <= 3 * 2.0 ** -8 * size + 1e-30 * min(v_scale, 1.0)).all()), float((err / size.clamp_min(1e-30)).max())


@pytest.mark.parametrize("B2,N", [(1, 257), (2, 288), (3, 289), (2, 320), (5, 321), (1, 384), (3, 385), (2, 500), (1, 1030), (2, 1152)])
def test_edges(dev, B2, N):
    _case(dev, B2, 4, N, None, None)


# within the range of the zero reference; below and above it; a mixture, so that some waves of a workgroup are out of range
@pytest.mark.parametrize("shift", [(60.0,), (-60.0,), (-100.0,), (120.0,), (2048.0,), (-2048.0,), (0.0, 0.0, -512.0, 0.0, 64.0, 512.0)])
def test_scores_far_from_zero(dev, shift):
    _case(dev, 3, 2, 300, shift, None)


# sums of probabilities within range whose products with v are not: beyond the largest number, and below the smallest normal one; and
# values of the same size beside sums of the other kind
@pytest.mark.parametrize("shift,v_scale", [((60.0,), 1e30), ((-60.0,), 1e-25), ((-75.0,), 1e-30), ((90.0, 0.0), 1e15), ((60.0,), 1e-30), ((-60.0,), 1e30)])
def test_values_far_from_one(dev, shift, v_scale):
    _case(dev, 3, 2, 300, shift, None, v_scale)


def test_a_second_walk_changes_the_queries_that_need_it_only(dev):
    """Scores out of range in some queries and values too large for another batch row's sums: everyone else's bits stay."""
    from fastfold_amd import _lib
    from fastfold_amd.model.fastnn.kernel import layouts
    g = torch.Generator().manual_seed(11)
    B2, H, N = 4, 2, 300
    q, k, v = (torch.randn(B2, H, N, 32, generator=g).to(BF).to(dev) for _ in range(3))
    bias = (torch.randn(H, N, N, generator=g) * 2).to(BF).to(dev)
    kb, fl = torch.empty(B2, layouts.n_tiles(N) * 32, device=dev), torch.empty(B2, layouts.n_tiles(N), dtype=torch.int32, device=dev)
    _lib.key_bias(kb, fl, None, B=B2, N=N)

    def run(v, bias):
        out = torch.empty(B2, N, H, 32, dtype=BF, device=dev)
        _lib.attention_fwd(out, layouts.tile_qk(q), layouts.tile_qk(k), layouts.tile_v(v), layouts.tile_bias(bias), kb, fl, None, B2=B2, H=H,
                           Nq=N, Nk=N)
        torch.cuda.synchronize()
        return out
    far = torch.zeros(N, dtype=torch.bool, device=dev)
    far[[5, 40, 41, 131, 299]] = True
    bias[:, far] = (bias[:, far] / 4).round() * 4               # 512 more or less of them is exact
    first, v2, bias2 = run(v, bias), v.clone(), bias.clone()
    bias2[0, far] = bias2[0, far] + 512.0
    v2[3, 1] = v2[3, 1] * 2.0 ** 124                            # sums of a few hundred such values overflow
    second = run(v2, bias2)
    assert torch.equal(second[:, ~far, 0], first[:, ~far, 0]) and torch.equal(second[:3, :, 1], first[:3, :, 1])
    # ... and those that were walked again are right: softmax takes no notice of what is added to a whole row
    near = second[:, far, 0].float() - first[:, far, 0].float()
    # (probabilities and results rounded to bf16 on either side, scores of 512 to 2^-14)
    assert float(near.norm()) <= (2 * 2.0 ** -8 + 2.0 ** -13) * float(first[:, far, 0].float().norm())
    assert bool(second.isfinite().all())


@pytest.mark.parametrize("N", [270, 400])
def test_masks(dev, N):
    g = torch.Generator().manual_seed(N)
    mask = (torch.rand(6, N, generator=g) > 0.3).float()
    mask[1] = 0                                              # no key at all, beside a row with keys
    mask[2, :-3], mask[3, 5:] = 0, 0
    mask[4:] = 0                                             # a pair of rows without keys
    _case(dev, 6, 4, N, None, mask)
