"""Ragged extents in bf16: the stacks run zero-padded to whole 32-row tiles; checked against the same modules in fp32,
which run at the extents as they are."""
import copy

import pytest
import torch

pytestmark = pytest.mark.gpu


def _init(mod, dev):
    g = torch.Generator().manual_seed(3)
    with torch.no_grad():
        for n, p in mod.named_parameters():
            w = torch.randn(p.shape, generator=g) * (0.1 if p.dim() == 1 else p.shape[-1] ** -0.5)
            p.copy_(1 + w if "norm" in n and n.endswith("weight") else w)
    return mod.to(dev).eval()


def _rel(a, b):
    return float((a.float() - b.float()).norm() / b.float().norm())


def _inputs(dev, s, r, c_m, pad):
    g = torch.Generator().manual_seed(100 * s + r)
    m, z = (torch.randn(*sh, generator=g).to(dev, torch.bfloat16) for sh in ((s, r, c_m), (r, r, 128)))
    res = torch.ones(r, device=dev)
    res[r - pad:] = 0 if pad else 1
    return m, z, (torch.ones(s, 1, device=dev) * res).bfloat16(), (res[:, None] * res).bfloat16()


@pytest.mark.parametrize("s,r,pad", [(1, 1, 0), (5, 31, 2), (32, 33, 0), (33, 64, 5), (65, 95, 0), (129, 40, 3)])
def test_trunk_at_ragged_extents(dev, s, r, pad):
    from fastfold_amd.model.fastnn import EvoformerStack
    fast = _init(EvoformerStack(256, 128, 384, 2, 1), dev)
    m, z, mm, pm = _inputs(dev, s, r, 256, pad)
    nv = r - pad
    with torch.no_grad():
        rm, rz, rs = fast(m.float(), z.float(), mm.float(), pm.float())
        half = copy.deepcopy(fast).bfloat16()
        m0, z0 = m.clone(), z.clone()
        gm, gz, gs = half(m, z, mm, pm)
        assert torch.equal(m, m0) and torch.equal(z, z0)
        lm, lz = [m.clone()], [z.clone()]
        own = (lm[0].data_ptr(), lz[0].data_ptr())
        _, _, ls = half.inplace(lm, lz, mm, pm)
    assert gm.shape == rm.shape and gz.shape == rz.shape and gs.shape == rs.shape
    assert _rel(gm[:, :nv], rm[:, :nv]) < 2e-2 and _rel(gz[:nv, :nv], rz[:nv, :nv]) < 2e-2 and _rel(gs[:nv], rs[:nv]) < 2e-2
    assert (lm[0].data_ptr(), lz[0].data_ptr()) == own           # updated where they are
    assert torch.equal(lm[0], gm) and torch.equal(lz[0], gz) and torch.equal(ls, gs)


@pytest.mark.parametrize("s,r", [(3, 33), (40, 31)])
def test_block_dropout_multipliers_at_ragged_extents(dev, s, r):
    """The multipliers of a training-mode forward apply at the padded extents too, in place and out of place."""
    from fastfold_amd.model.fastnn import Evoformer
    blk = _init(Evoformer(256, 128, True, True), dev).train()
    m, z, mm, pm = _inputs(dev, s, r, 256, 0)
    with torch.no_grad():
        drops = blk._draw_drops(m[None].float(), z[None].float())
        rm, rz = blk._core(m[None].float(), z[None].float(), mm[None].float(), pm[None].float(), False, drops=drops)
        half = copy.deepcopy(blk).bfloat16()
        d16 = {k: v.bfloat16() for k, v in drops.items()}
        gm, gz = half._core_any(m[None], z[None], mm[None], pm[None], False, drops=d16)
        im, iz = half._core_any(m[None].clone(), z[None].clone(), mm[None], pm[None], True, drops=d16)
    assert _rel(gm, rm) < 2e-2 and _rel(gz, rz) < 2e-2
    assert torch.equal(im, gm) and torch.equal(iz, gz)


@pytest.mark.parametrize("s,r", [(7, 33), (70, 45)])
def test_feeder_stacks_at_ragged_extents(dev, s, r):
    from fastfold_amd.model.fastnn import ExtraMSAStack, TemplatePairStack
    ex = _init(ExtraMSAStack(64, 128, 2), dev)
    m, z, mm, pm = _inputs(dev, s, r, 64, 3)
    tp = _init(TemplatePairStack(64, 16, 64, 2, 4, 2, 0.25, None), dev)
    t = torch.randn(2, r, r, 64, device=dev).bfloat16()
    nv = r - 3
    with torch.no_grad():
        ref = ex(m.float(), z.float(), None, mm.float(), pm.float())
        out = copy.deepcopy(ex).bfloat16()(m, z, None, mm, pm)
        assert _rel(out[:nv, :nv], ref[:nv, :nv]) < 2e-2
        ref = tp(t.float(), pm[None].float(), None)
        half = copy.deepcopy(tp).bfloat16()
        out = half(t, pm[None], None)
        assert _rel(out[:, :nv, :nv], ref[:, :nv, :nv]) < 2e-2
        lst = [t.clone()]
        half.inplace(lst, pm[None], None)
        assert torch.equal(lst[0], out)


@pytest.mark.parametrize("r", [32, 45])
def test_under_inference_mode(dev, r):
    """Stacks and single blocks with masks from outside and with masks made under ``torch.inference_mode``, which have no version
    counter (the padded ones of a ragged bf16 call are always such): the bits of the call under ``torch.no_grad``."""
    from fastfold_amd.model.fastnn import Evoformer, EvoformerStack, ExtraMSABlock, ExtraMSAStack, TemplatePairStack
    m, z, mm, pm = _inputs(dev, 33, r, 256, 3)
    e = m[..., :64].contiguous()
    t = torch.randn(2, r, r, 64, device=dev).bfloat16()
    mods = [(_init(mod, dev).bfloat16(), call) for mod, call in (
        (EvoformerStack(256, 128, 384, 2, 1), lambda f, a, b: f(m, z, a, b)),
        (Evoformer(256, 128, True, True), lambda f, a, b: f(m, z, a, b)),
        (ExtraMSAStack(64, 128, 2), lambda f, a, b: (f(e, z, None, a, b),)),
        (ExtraMSABlock(64, 128, True, True), lambda f, a, b: f(e, z, a, b)),
        (TemplatePairStack(64, 16, 64, 2, 4, 2, 0.25, None), lambda f, a, b: (f(t, b[None], None),)))]
    for mod, call in mods:
        with torch.no_grad():
            want = call(mod, mm, pm)
        with torch.inference_mode():
            for a, b in ((mm, pm), (mm.clone(), pm.clone()), (mm.clone(), pm.clone())):
                got = call(mod, a, b)
                assert all(torch.equal(x, y) for x, y in zip(got, want)), type(mod).__name__
        with torch.no_grad():
            assert all(torch.equal(x, y) for x, y in zip(call(mod, mm, pm), want))


@pytest.mark.parametrize("kind", ["trunk", "extra"])
def test_in_place_memory_at_ragged_extents(dev, kind, monkeypatch):
    """The padded copies of an in-place call take no more than the un-padded run takes in gate tensors and unfused scratch (5 %
    of the peak beyond the inputs), and no more than themselves beyond the peak at the next whole tile."""
    from fastfold_amd.model.fastnn import EvoformerStack, ExtraMSAStack, _fused, set_chunk_size
    s, r = 64, 1270
    mod = _init(EvoformerStack(256, 128, 384, 1, 1) if kind == "trunk" else ExtraMSAStack(64, 128, 1), dev).bfloat16()
    c_m = 256 if kind == "trunk" else 64

    def peak(r):
        m, z, mm, pm = _inputs(dev, s, r, c_m, 3)
        with torch.no_grad():
            for _ in range(2):                                   # packs the weights; measured
                torch.cuda.synchronize()
                base = torch.cuda.memory_allocated()
                torch.cuda.reset_peak_memory_stats()
                mod.inplace([m], [z], mm, pm) if kind == "trunk" else mod.inplace([m], [z], None, mm, pm)
        torch.cuda.synchronize()
        return torch.cuda.max_memory_allocated() - base
    set_chunk_size(64)
    try:
        padded, whole = peak(r), peak(1280)
        monkeypatch.setattr(_fused, "pad_to_tiles", lambda m, z, mk, pk, pad_s=True: (m, z, mk, pk))
        as_it_is = peak(r)
    finally:
        set_chunk_size(None)
    assert padded <= 1.05 * as_it_is, (padded, as_it_is)
    assert padded <= whole + 1.02 * 2 * (s * 1280 * c_m + 1280 * 1280 * 128), (padded, whole)
