"""Launch plans: a replayed block gives the bits of the Python launch sequence, follows its parameters, and works on any
stream and from several threads; ``ffk_run_plan`` refuses malformed plans on the host."""
import copy
import ctypes
import struct
import threading

import pytest
import torch

gpu = pytest.mark.gpu


def _stack(dev, dtype, n=2):
    from fastfold_amd.model.fastnn import EvoformerStack
    g = torch.Generator().manual_seed(1)
    st = EvoformerStack(256, 128, 384, n, 1)
    with torch.no_grad():
        for p in st.parameters():
            p.copy_(torch.randn(p.shape, generator=g) * 0.1)
    return st.to(dev, dtype).eval()


def _inputs(dev, dtype, s, r, seed):
    g = torch.Generator().manual_seed(seed)
    m, z = torch.randn(s, r, 256, generator=g).to(dev, dtype), torch.randn(r, r, 128, generator=g).to(dev, dtype)
    res = (torch.rand(r, generator=g) > 0.2).float().to(dev, dtype)
    return m, z, torch.ones(s, 1, device=dev, dtype=dtype) * res, res[:, None] * res


def _in_python(fn):
    """fn() with every launch issued from Python (timing records exist)."""
    from fastfold_amd import _lib
    _lib.time_kernel("ffk_softmax_fwd")
    try:
        return fn()
    finally:
        _lib.time_kernel("ffk_softmax_fwd", enable=False)


@gpu
@pytest.mark.parametrize("dtype,s,r,multimer", [(torch.bfloat16, 64, 64, False), (torch.bfloat16, 5, 33, False),
                                                (torch.float32, 5, 33, False), (torch.bfloat16, 160, 96, True)])
def test_replay_gives_the_bits_of_the_sequence(dev, dtype, s, r, multimer):
    st = _stack(dev, dtype)
    for b in st.blocks:
        b.is_multimer = multimer
    with torch.no_grad():
        for seed in range(4):                # packs weights, records, replays, replays
            x = _inputs(dev, dtype, s, r, seed)
            got = st(*x)
            want = _in_python(lambda: st(*x))
            assert all(torch.equal(a, b) for a, b in zip(got, want)), seed
    plans = st.blocks[1].__dict__["_plan_state"].plans
    assert len(plans) == 1 and next(iter(plans.values())).blob


@gpu
def test_replay_follows_the_parameters(dev):
    st = _stack(dev, torch.bfloat16, 1)
    x = _inputs(dev, torch.bfloat16, 32, 32, 0)
    blk = st.blocks[0]

    def check():
        with torch.no_grad():
            got, want = st(*x), _in_python(lambda: st(*x))
        assert all(torch.equal(a, b) for a, b in zip(got, want))
        return got[1]
    with torch.no_grad():
        for _ in range(3):
            z0 = check()
        blk.pair.PairTransition.linear2.weight.mul_(2.0)                       # in place
        z1 = check()
        assert not torch.equal(z0, z1)
        check()
        blk.pair.PairTransition.linear2.weight.data.mul_(2.0)                  # behind the version counter
        blk.pair.PairTransition.invalidate_packed()
        z2 = check()
        assert not torch.equal(z1, z2)
        check()
        blk.pair.PairTransition = copy.deepcopy(_stack(dev, torch.bfloat16, 1).blocks[0].pair.PairTransition)   # exchanged
        assert torch.equal(check(), z0)
        other = copy.deepcopy(st)                                              # a copy plans for itself
        other.blocks[0].pair.PairTransition.linear2.weight.zero_()
        assert torch.equal(check(), z0) and not torch.equal(other(*x)[1], z0)


@gpu
def test_replay_from_several_threads_and_streams(dev):
    st = _stack(dev, torch.bfloat16)
    xs = [_inputs(dev, torch.bfloat16, 32, 64, k) for k in range(4)]
    with torch.no_grad():
        want = [[t.clone() for t in st(*x)] for x in xs]
    torch.cuda.synchronize()
    bad = []

    def guarded(k):
        try:
            work(k)
        except Exception as e:
            bad.append((k, repr(e)))

    def work(k):
        side = torch.cuda.Stream()
        with torch.no_grad(), torch.cuda.stream(side):
            for _ in range(6):
                got = st(*xs[k])
                side.synchronize()
                if not all(torch.equal(a, b) for a, b in zip(got, want[k])):
                    bad.append(k)
    threads = [threading.Thread(target=guarded, args=(k,)) for k in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not bad, bad


def test_malformed_plans_are_refused():
    from fastfold_amd import _lib
    lib = _lib.load()
    bases = (ctypes.c_uint64 * 2)(0, 0)

    def run(blob):
        return lib.ffk_run_plan(blob, len(blob), bases, 2, None)
    assert run(b"") == 0
    assert run(b"\0" * 8) == 2                                                           # shorter than a head
    assert run(struct.pack("<iiii", 99, 2, 0, 0) + b"\0" * 16) == 2                      # no such operation
    assert run(struct.pack("<iiii", 9, 1, 0, 0) + b"\0" * 8) == 2                        # wrong number of arguments
    assert run(struct.pack("<iiii", 9, 2, 1, 0) + struct.pack("<iiq", 0, 7, 0) + b"\0" * 16) == 2      # no such buffer
    assert run(struct.pack("<iiii", 9, 2, 1, 0) + struct.pack("<iiq", 0, 1, 0) + b"\0" * 16) == 2      # a null buffer
    assert run(struct.pack("<iiii", 9, 2, 0, 0) + struct.pack("<Qq", 0, 16)) == 3        # the entry point's own check


@gpu
@pytest.mark.parametrize("s,r", [(12, 40), (16, 64)])
def test_replay_under_memory_of_any_content(dev, s, r):
    """Forward and backward of a block with freshly filled memory around (zeros, NaN): recorded and replayed passes give the
    same bits, so no launch reads scratch it has not written and no replay takes a neighbour's buffer."""
    from fastfold_amd.model.fastnn import Evoformer
    st = _stack(dev, torch.bfloat16, 1)
    blk = Evoformer(256, 128, True, True).to(dev, torch.bfloat16)
    blk.load_state_dict(st.blocks[0].state_dict())
    blk.train()
    m, z, mm, pm = _inputs(dev, torch.bfloat16, s, r, 3)
    cot = torch.randn(s, r, 256, device=dev).bfloat16(), torch.randn(r, r, 128, device=dev).bfloat16()
    want = None
    for fill in (0.0, float("nan"), float("nan"), float("nan")):
        torch.cuda.synchronize()
        torch.cuda.empty_cache()
        junk = [torch.full((n,), fill, device=dev) for n in [1 << 25] * 2 + [1 << 18] * 64 + [1 << 12] * 200]
        del junk
        torch.manual_seed(5)
        a, b = m.clone().requires_grad_(), z.clone().requires_grad_()
        for p in blk.parameters():
            p.grad = None
        out = blk(a, b, mm, pm)
        torch.autograd.backward(out, cot)
        got = [*out, a.grad, b.grad, *(p.grad for p in blk.parameters())]
        got = [t.detach().clone() for t in got]
        assert all(bool(torch.isfinite(t).all()) for t in got)
        if want is not None:
            assert all(torch.equal(x, y) for x, y in zip(got, want))
        want = got


@gpu
@pytest.mark.parametrize("kind,dtype", [("evoformer", torch.float32), ("evoformer", torch.bfloat16), ("extra", torch.bfloat16),
                                        ("backward", torch.float32)])
def test_replay_with_other_buffers_shared(dev, kind, dtype):
    """s == r, so that both masks have one shape: a block recorded with one tensor as both masks (and, backward, the input as
    the cotangent), then called with two; and the other way round."""
    from fastfold_amd.model.fastnn import Evoformer, ExtraMSABlock
    n = 64
    st = _stack(dev, dtype, 1)
    if kind == "extra":
        g = torch.Generator().manual_seed(2)
        blk = ExtraMSABlock(64, 128, True, True)
        with torch.no_grad():
            for p in blk.parameters():
                p.copy_(torch.randn(p.shape, generator=g) * 0.1)
        blk = blk.to(dev, dtype).eval()
    else:
        blk = Evoformer(256, 128, True, True).to(dev, dtype).eval()
        blk.load_state_dict(st.blocks[0].state_dict())
    m, z, mm, pm = _inputs(dev, dtype, n, n, 7)
    m = m[..., :64].contiguous() if kind == "extra" else m
    ones = torch.ones_like(pm)
    dm, dz = torch.randn_like(m), torch.randn_like(z)

    def call(msa_mask, pair_mask, own_cotangent):
        if kind != "backward":
            with torch.no_grad():
                return blk(m, z, msa_mask, pair_mask)
        with torch.no_grad():
            a, b = m[None], z[None]
            cot = (a, b) if own_cotangent else (dm[None], dz[None])
            da, db, grads = blk._backward(a, b, msa_mask[None], pair_mask[None], *cot, None)
            return [da, db, *grads]
    for args in [(ones, ones, True)] * 3 + [(mm, pm, False)] * 3 + [(ones, ones, True), (mm, pm, True), (pm, mm, False)]:
        got = call(*args)
        want = _in_python(lambda: call(*args))
        assert all(torch.equal(x, y) for x, y in zip(got, want))
