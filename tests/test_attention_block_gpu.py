"""ffk_attention_block (a gated attention from the rows of x to the updated rows in one kernel) through the C ABI against float64
(fastfold/model/fastnn/ops.py:289-331), at the edges of its tiles, waves and layouts."""
import math

import pytest
import torch

pytestmark = pytest.mark.gpu
BF = torch.bfloat16
LOG2E = math.log2(math.e)


def _case(dev, C, D, B2, N, seed, transposed=False, bias=True):
    g = torch.Generator().manual_seed(seed)
    H = C // D

    def rnd(*shape, scale=1.0, shift=0.0):
        return (torch.randn(*shape, generator=g) * scale + shift).to(dev, BF)
    p = dict(C=C, D=D, H=H, B2=B2, N=N, qkv=rnd(3 * C, C, scale=C ** -0.5), wg=rnd(C, C, scale=C ** -0.5),
             bg=rnd(C), wo=rnd(C, C, scale=C ** -0.5), gam=rnd(C, scale=0.1, shift=1.0), bet=rnd(C, scale=0.1))
    p["x"] = rnd(N, B2, C, scale=1.5, shift=0.3).transpose(0, 1) if transposed else rnd(B2, N, C, scale=1.5, shift=0.3)
    p["bias"] = rnd(H, N, N, scale=1.5) if bias else None   # in the kernel's unit, log2: the same rounded numbers on both sides
    mask = torch.ones(B2, N)
    mask[0, N - N // 3:] = 0                                  # a masked tail
    if B2 > 1:
        mask[1] = (torch.rand(N, generator=g) > 0.3).float()  # masked keys in every tile
    if B2 > 2:
        mask[2] = 0                                           # no key at all
    if B2 > 3:
        mask[3, :min(32, N - 1)] = 0                          # a first tile without one
    p["mask"] = mask.to(dev, BF)
    return p


def _heads(p):
    """The gated heads in float64 from the rounded rows and operands that the kernel multiplies."""
    x = p["x"].double().cpu()
    mu = x.mean(-1, keepdim=True)
    y = (x - mu) / torch.sqrt(((x - mu) ** 2).mean(-1, keepdim=True) + 1e-5) * p["gam"].double().cpu() + p["bet"].double().cpu()
    y = y.to(BF).double()
    B2, N, C, H, D = (p[k] for k in ("B2", "N", "C", "H", "D"))
    q, k, v = (t.view(B2, N, H, D).transpose(1, 2) for t in (y @ p["qkv"].double().cpu().t()).split(C, -1))
    s = (q * D ** -0.5) @ k.transpose(-1, -2)
    if p["bias"] is not None:
        s = s + p["bias"].double().cpu() / LOG2E
    mask = p["mask"].double().cpu()
    s = s.masked_fill(mask[:, None, None, :] == 0, -1e9)
    o = (torch.softmax(s, -1) @ v).transpose(1, 2).reshape(B2, N, C)
    return torch.sigmoid(y @ p["wg"].double().cpu().t() + p["bg"].double().cpu()) * o


def _update(p, drop=None, bo=None):
    upd = _heads(p) @ p["wo"].double().cpu().t()
    upd = upd + (0 if bo is None else bo.double().cpu())
    return upd * (1 if drop is None else drop.double().cpu())


def _run(p, x, out, bo=None, drop=None, xtail=None):
    from fastfold_amd import _lib
    from fastfold_amd.model.fastnn import _fused as F_
    from fastfold_amd.model.fastnn.kernel import layouts
    dev, B2, N, C = x.device, p["B2"], p["N"], p["C"]
    w = F_.pack_attention_block(p["qkv"], p["wg"], p["wo"], BF, dev)
    bias = None if p["bias"] is None else layouts.tile_bias(p["bias"])
    kb, flags = F_.key_bias(p["mask"], dev, B2=B2, N=N, mask_sb=N, mask_sn=1)
    _lib.attention_block(out, x, p["gam"], p["bet"], w, p["bg"], bo, bias, kb, flags, B2=B2, N=N, C=C, D=p["D"],
                         s_row=x.stride(0), s_tok=x.stride(1), bias_pitch=(N + 31) // 32, xtail=xtail, drop=drop)
    torch.cuda.synchronize()


def _stream(h, tail):
    """The 24-bit values of an extended residual stream."""
    return ((h.view(torch.int16).to(torch.int32) << 16) + (tail.to(torch.int32) << 8)).view(torch.float32)


def _err(got, p, upd, live=slice(None)):
    d = (got.double().cpu() - p["x"].double().cpu())[live] - upd[live]
    return float(d.norm() / upd[live].norm())


# Six roundings to bf16 in a chain (q or k, v, p, o, gated o, update), each by at most 2^-9 of a value.  The result is read at 24 bits:
# its rounding to bf16 would be one of the stream, which is several times as large as the update.
TOL = 6 * 2.0 ** -9


# One tile per wave with its heads divided by four, two and not at all; several tiles per wave; ragged rows; more batch rows than
# a multiple of eight.
@pytest.mark.parametrize("C,D,N", [(128, 32, n) for n in (1, 32, 50, 64, 96, 128, 129, 160, 224, 256)]
                         + [(64, 16, n) for n in (32, 77, 128, 160, 256, 288, 320, 500, 512)]
                         + [(64, 8, n) for n in (20, 32, 96, 128, 200, 256, 257, 384)]
                         + [(256, 32, n) for n in (5, 32, 64, 65, 96, 128)] + [(256, -32, n) for n in (32, 50, 96, 128)])
def test_attention_block_against_float64(dev, C, D, N):
    p = _case(dev, C, abs(D), 9, N, seed=C + N, transposed=N % 3 == 0, bias=C != 256 or D < 0)
    out = torch.empty_like(p["x"])                            # keeps the strides
    tail = torch.empty_like(out, dtype=torch.int8).zero_()
    _run(p, p["x"], out, xtail=tail)
    live = [0, 1] + list(range(3, 9))                         # all keys masked: what the reference averages over is arbitrary
    assert _err(_stream(out, tail), p, _update(p), live) < TOL
    # ... and the heads are zero here, so that the row stays as it was
    assert torch.equal(out[2], p["x"][2])


@pytest.mark.parametrize("C,D,N", [(128, 32, 96), (128, 32, 256), (64, 16, 320), (64, 8, 160), (256, 32, 128)])
def test_attention_block_residual_forms(dev, C, D, N):
    """Output bias, dropout multipliers, in place, and the tail of an extended residual stream."""
    p = _case(dev, C, D, 3, N, seed=N, bias=C != 256)
    p["mask"][2] = 1
    g = torch.Generator().manual_seed(1)
    bo = torch.randn(C, generator=g).to(dev, BF)
    drop = ((torch.rand(N, C, generator=g) > 0.25).float() / 0.75).to(dev, BF)
    want = _update(p, drop, bo)
    plain = torch.empty_like(p["x"])
    _run(p, p["x"], plain, bo, drop)
    x2, tail = p["x"].clone(), torch.zeros(p["x"].shape, dtype=torch.int8, device=dev)
    _run(p, x2, x2, bo, drop, tail)
    # half up against half to even: one bf16 step at most
    assert float(((x2.float() - plain.float()).abs() / plain.float().abs().clamp_min(1e-3)).max()) <= 2.0 ** -7
    assert _err(_stream(x2, tail), p, want) < TOL


@pytest.mark.parametrize("C,D", [(128, 32), (64, 16), (64, 8)])
def test_attention_block_moving_reference(dev, C, D):
    """Scores that rise far above those of the first tile: the second walk, with the reference moved tile by tile."""
    p = _case(dev, C, D, 4, 256, seed=2)
    p["mask"][:] = 1
    rise = torch.arange(8, device=dev).repeat_interleave(32).float() * 80.0
    p["bias"] = (p["bias"].float() + rise[None, None, :]).to(BF)
    p["bias"][:, 100:140] = p["bias"][:, 100:140].flip(-1)    # ... and falling ones in the same tiles of queries
    out = p["x"].clone()
    tail = torch.zeros(out.shape, dtype=torch.int8, device=dev)
    _run(p, out, out, xtail=tail)
    assert _err(_stream(out, tail), p, _update(p)) < TOL


@pytest.mark.parametrize("N", [32, 100, 129, 160, 192, 225, 256])
def test_attention_heads_against_float64(dev, N):
    from fastfold_amd import _lib
    from fastfold_amd.model.fastnn import _fused as F_
    from fastfold_amd.model.fastnn.kernel import layouts
    p = _case(dev, 256, 32, 5, N, seed=N, transposed=N % 2 == 1)
    kb, flags = F_.key_bias(p["mask"], dev, B2=5, N=N, mask_sb=N, mask_sn=1)
    o = torch.full((5, N, 256), float("nan"), device=dev, dtype=BF)
    _lib.attention_heads(o, p["x"], p["gam"], p["bet"], F_.pack_attention_block(p["qkv"], p["wg"], p["wo"], BF, dev), p["bg"],
                         layouts.tile_bias(p["bias"]), kb, flags, B2=5, N=N, C=256, D=32, s_row=p["x"].stride(0),
                         s_tok=p["x"].stride(1), bias_pitch=(N + 31) // 32)
    torch.cuda.synchronize()
    want = _heads(p)
    live = [0, 1, 3, 4]
    assert float((o.double().cpu() - want)[live].norm() / want[live].norm()) < TOL
    assert float(o[2].abs().max()) == 0.0                     # no key at all


@pytest.mark.parametrize("N", [64, 96, 160, 200, 224, 256])
def test_the_gate_of_128_channels_is_not_rounded_ahead_of_its_product(dev, N):
    """Uniform attention over equal exact values and an output projection that is the identity: one rounding to bf16, of gate times
    value, is all that happens."""
    C, v = 128, 1.1015625
    g = torch.Generator().manual_seed(N)
    eye = torch.eye(C)
    p = dict(C=C, D=32, H=4, B2=3, N=N, qkv=torch.cat([torch.zeros(2 * C, C), eye]).to(dev, BF), wg=torch.zeros(C, C, device=dev, dtype=BF),
             bg=torch.randn(C, generator=g).to(dev, BF), wo=eye.to(dev, BF), gam=torch.zeros(C, device=dev, dtype=BF),
             bet=torch.full((C,), v, device=dev, dtype=BF), x=torch.zeros(3, N, C, device=dev, dtype=BF),
             bias=torch.zeros(4, N, N, device=dev, dtype=BF), mask=torch.ones(3, N, device=dev, dtype=BF))
    out = torch.empty_like(p["x"])
    _run(p, p["x"], out)
    want = torch.sigmoid(p["bg"].double().cpu()) * v
    # half a step of the result, and 2^-20 for the fp32 exponential, reciprocals and mean
    assert bool(((out.double().cpu() - want).abs() <= (2.0 ** -9 + 2.0 ** -20) * 2.0 ** want.log2().floor() * 2).all())


def test_attention_block_refuses(dev):
    p = _case(dev, 256, 32, 2, 129, seed=0)
    with pytest.raises(RuntimeError, match="too long"):
        _run(p, p["x"], torch.empty_like(p["x"]))
    p = _case(dev, 128, 32, 2, 257, seed=0)
    with pytest.raises(RuntimeError, match="too long"):
        _run(p, p["x"], torch.empty_like(p["x"]))
    p = _case(dev, 128, 32, 2, 64, seed=0, bias=False)
    with pytest.raises(RuntimeError, match="pair bias"):
        _run(p, p["x"], torch.empty_like(p["x"]))


def _modules(dev):
    from fastfold_amd.model.fastnn.msa import MSAColumnAttention, MSARowAttentionWithPairBias
    from fastfold_amd.model.fastnn.ops import ChunkTriangleAttentionEndingNode, ChunkTriangleAttentionStartingNode

    def pair(r, c, **kw):
        z, pm = torch.randn(1, r, r, c, device=dev).to(BF), torch.ones(1, r, r, device=dev, dtype=BF)
        pm[:, -5:] = 0
        pm[:, :, -5:] = 0
        return z, pm

    def msa(s, r, c):
        m, mm = torch.randn(1, s, r, c, device=dev).to(BF), torch.ones(1, s, r, device=dev, dtype=BF)
        mm[:, :, -5:] = 0
        return m, mm
    for r, c, d in ((64, 128, 32), (160, 128, 32), (96, 64, 16)):
        for cls in (ChunkTriangleAttentionStartingNode, ChunkTriangleAttentionEndingNode):
            yield cls(c, 0.25, c=d, n_head=4), pair(r, c)
    for s, r, c, d in ((64, 96, 256, 32), (60, 160, 256, 32), (40, 96, 64, 8)):
        m, mm = msa(s, r, c)
        yield MSARowAttentionWithPairBias(c, 128, c=d, n_head=8), (m, pair(r, 128)[0], mm)
    yield MSAColumnAttention(256), msa(96, 64, 256)


def test_modules_take_the_block_and_match_the_separate_launches(dev, monkeypatch):
    """Every attention module at sizes that go to the one kernel, against the same module as projection, core and output stage: the two
    differ by their own bf16 roundings only (six of 2^-9 on either side)."""
    from fastfold_amd import _lib
    from fastfold_amd.model.fastnn import _fused as F_
    torch.manual_seed(4)
    names, call = [], _lib.call
    monkeypatch.setattr(_lib, "call", lambda name, *a: (names.append(name), call(name, *a))[1])
    for mod, args in _modules(dev):
        with torch.no_grad():
            for n, p in mod.named_parameters():
                p.copy_(1 + 0.1 * torch.randn_like(p) if "layernorm" in n and n.endswith("weight")
                        else torch.randn_like(p) * (0.3 if p.dim() == 1 else p.shape[-1] ** -0.5))
        mod = mod.to(dev, BF).eval()
        outs = []
        for on in (True, False):
            monkeypatch.setattr(F_, "_ATTENTION_BLOCK", on)
            del names[:]
            with torch.no_grad():
                outs.append(mod(*args).float())
            assert on == any(n in ("ffk_attention_block", "ffk_attention_heads") for n in names), (type(mod).__name__, names)
        upd = outs[1] - args[0].float()
        err = float((outs[0] - outs[1]).norm() / upd.norm())
        assert float(upd.norm()) > 1.0 and err < 2 * TOL, (type(mod).__name__, args[0].shape, err)


@pytest.mark.parametrize("rows,tokens,C,D", [(300, 128, 256, 0), (200, 96, 256, 32), (256, 256, 256, 32), (512, 256, 64, 8)])
def test_a_subset_of_the_rows_gives_the_bits_of_all(dev, rows, tokens, C, D):
    """Column attention (D = 0) and row attention of few rows, a single one and all of them."""
    from fastfold_amd.model.fastnn.msa import MSAColumnAttention, MSARowAttentionWithPairBias
    torch.manual_seed(tokens)
    mod = MSAColumnAttention(C) if D == 0 else MSARowAttentionWithPairBias(C, 128, c=D, n_head=C // D)
    with torch.no_grad():
        for n, p in mod.named_parameters():
            p.copy_(1 + 0.1 * torch.randn_like(p) if "layernorm" in n and n.endswith("weight")
                    else torch.randn_like(p) * (0.3 if p.dim() == 1 else p.shape[-1] ** -0.5))
    mod = mod.to(dev, BF).eval()
    m = torch.randn(1, rows, tokens, C, device=dev).to(BF)
    mask = (torch.rand(1, rows, tokens, device=dev) > 0.2).to(BF)
    z = torch.randn(1, tokens, tokens, 128, device=dev).to(BF)

    def run(m, mask):
        with torch.no_grad():
            return mod(m.transpose(1, 2).contiguous(), mask.transpose(1, 2).contiguous()).transpose(1, 2) if D == 0 else mod(m, z, mask)
    full = run(m, mask)
    assert float((full - m).float().abs().max()) > 0.1
    for lo, hi in ((5, 36), (0, 1), (rows - 60, rows)):
        assert torch.equal(run(m[:, lo:hi].contiguous(), mask[:, lo:hi].contiguous()), full[:, lo:hi]), (lo, hi)


def test_weights_of_short_rows_are_laid_out_with_the_others(dev):
    """The first pass of a triangle attention lays out all weights: the first pass at a length that takes another route builds
    nothing, so a stack can record it."""
    from fastfold_amd import _plan
    from fastfold_amd.model.fastnn.ops import ChunkTriangleAttentionStartingNode
    torch.manual_seed(0)
    att = ChunkTriangleAttentionStartingNode(128, 32).to(dev, BF).eval()
    with torch.no_grad():
        for i, r in enumerate((288, 64, 256)):
            z = torch.randn(1, r, r, 128, device=dev, dtype=BF)
            before = _plan.builds
            out = att(z, torch.ones(1, r, r, device=dev, dtype=BF))
            assert bool(out.isfinite().all()) and (i == 0 or _plan.builds == before)


def test_modules_with_normalisation_weights_anywhere(dev):
    """LayerNorm parameters that are slices of a flat buffer, not on 16 bytes: the same update by the launches that take them (six
    roundings of 2^-9 on either side; a transition has three)."""
    from fastfold_amd.model.fastnn.kernel import LayerNorm
    from fastfold_amd.model.fastnn.ops import Transition
    torch.manual_seed(5)
    cases = list(_modules(dev)) + [(Transition(64), (torch.randn(1, 40, 96, 64, device=dev).to(BF),))]
    for mod, args in cases:
        with torch.no_grad():
            for n, p in mod.named_parameters():
                p.copy_(1 + 0.1 * torch.randn_like(p) if "norm" in n and n.endswith("weight")
                        else torch.randn_like(p) * (0.3 if p.dim() == 1 else p.shape[-1] ** -0.5))
        mod = mod.to(dev, BF).eval()
        outs = []
        for shift in (0, 1):
            for m in mod.modules():
                if isinstance(m, LayerNorm) and shift:
                    for p in (m.weight, m.bias):
                        flat = torch.zeros(p.numel() + 8, device=dev, dtype=BF)
                        flat[1:p.numel() + 1] = p.detach()
                        p.data = flat[1:p.numel() + 1]
            with torch.no_grad():
                outs.append(mod(*args).float())
        upd = outs[0] - args[0].float()
        assert float((outs[0] - outs[1]).norm() / upd.norm()) < 2 * TOL, (type(mod).__name__, args[0].shape)


@pytest.mark.parametrize("r", [32, 96, 128])
def test_triangle_attention_of_256_channels(dev, r):
    """Its pair bias is made by no kernel of 64 or 128 channels: launches of their own, against float64."""
    from fastfold_amd.model.fastnn.ops import ChunkTriangleAttentionStartingNode
    torch.manual_seed(r)
    mod = ChunkTriangleAttentionStartingNode(256, 0.25, c=32, n_head=8)
    with torch.no_grad():
        for n, p in mod.named_parameters():
            p.copy_(1 + 0.1 * torch.randn_like(p) if "norm" in n and n.endswith("weight")
                    else torch.randn_like(p) * (0.3 if p.dim() == 1 else p.shape[-1] ** -0.5))
    mod = mod.to(dev, BF).eval()
    z = torch.randn(1, r, r, 256, device=dev).to(BF)
    with torch.no_grad():
        got = mod(z, torch.ones(1, r, r, device=dev, dtype=BF)).double().cpu()
    d = lambda t: t.detach().double().cpu()                   # noqa: E731
    x = d(z)[0]
    y = torch.nn.functional.layer_norm(x, (256,), d(mod.layernorm1.weight), d(mod.layernorm1.bias))
    a = mod.attention
    q, k, v = (t.view(r, r, 8, 32).transpose(1, 2) for t in (y @ d(a.to_qkv.weight).t()).split(256, -1))
    s = q * 32 ** -0.5 @ k.transpose(-1, -2) + (y @ d(mod.linear_b.weight).t()).permute(2, 0, 1)
    o = (torch.softmax(s, -1) @ v).transpose(1, 2).reshape(r, r, 256)
    upd = (torch.sigmoid(y @ d(a.gating_linear.weight).t() + d(a.gating_bias)) * o) @ d(a.o_linear.weight).t() + d(mod.out_bias)
    # seven roundings of the update (y among them) and that of the result
    assert float((got[0] - x - upd).norm()) < 7 * 2.0 ** -9 * float(upd.norm()) + 2.0 ** -9 * float((x + upd).norm())
