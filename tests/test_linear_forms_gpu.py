"""ffk_fused_linear over the forms its descriptor has: random launches - row-major, strided, transposed and channel-major operands,
every tile kind with every epilogue it takes, whole and broken extents, several tiles of different kinds in a launch - against a
float64 model that addresses every element by the formulas of include/ffk.h.  Whichever kernel takes a launch, the elements of its
tiles have their values and no other element of the output buffers changes."""
import random

import numpy as np
import pytest
import torch

from oracle import ops_np

pytestmark = pytest.mark.gpu

STRIDED, QK, V, BIAS, ACC = range(5)
NONE, RELU, SIGMOID, GATE_POS = range(4)
TOL = {torch.float32: 2e-5, torch.bfloat16: 2e-2}      # of the largest value: 32-bit sums; two or three roundings to bf16
SIZES = [(1, 1), (3, 37), (3, 37), (5, 48), (5, 48), (40, 32), (40, 32), (70, 96), (131, 33), (333, 96)]


def _qk(n, d):
    return (d >> 4) * 512 + n * 16 + (d & 15)


def _acc(row, col):
    return ((((row & 7) >> 2) * 32 + col) << 4) + 4 * (row >> 3) + (row & 3)


def _offsets(t, M):
    """Element offsets [M, ncols] of a tile."""
    m, c = np.arange(M)[:, None], np.arange(t["ncols"])[None, :]
    hi, lo = m // t["inner"], m % t["inner"]
    head = hi * t["s_o"] + (c >> 5) * t["s_h"]
    if t["kind"] == STRIDED:
        return head + lo * t["s_i"] + (c & 31) * t["s_d"]
    if t["kind"] == BIAS:
        return c * t["s_h"] + (hi >> 5) * t["s_o"] + (lo >> 5) * 1024 + _qk(lo & 31, hi & 31)
    lo32, c32 = lo & 31, c & 31
    return head + (lo >> 5) * 1024 + (_qk(lo32, c32) if t["kind"] == QK else _acc(lo32, c32) if t["kind"] == V else _acc(c32, lo32))


def _form(r, bf16, K, chan):
    """A launch as plain values; strides of bf16 launches are multiples of 8 where the entry point asks for 16-byte rows."""
    B, N = r.choice(SIZES)
    v = 8 if bf16 else 4
    M = B * N - (r.randrange(N) if r.random() < 0.2 else 0)
    pad = lambda n, to: (n + to - 1) // to * to
    np_ = pad(N, r.choice([1, v, 16]))
    f = dict(M=M, K=K, ln=r.random() < 0.6, chan=chan)
    if chan:
        f.update(a_inner=N, **r.choice([dict(a_so=np_, a_si=1, a_cs=B * np_), dict(a_so=np_, a_si=1, a_cs=pad(B * np_, 8)), dict(a_so=1, a_si=B, a_cs=B * N)]))
    else:
        f.update(r.choice([dict(a_inner=M, a_so=0, a_si=K), dict(a_inner=0x7fffffff, a_so=0, a_si=K + 16), dict(a_inner=N, a_so=N * K, a_si=K),
                           dict(a_inner=N, a_so=K, a_si=B * K)]))
    kinds = r.choice([[STRIDED], [STRIDED, STRIDED], [ACC, QK, V, ACC], [V], [QK, V, STRIDED], [STRIDED, BIAS], [BIAS], [STRIDED, V, BIAS], ["cols", STRIDED], ["cols"]])
    same_mask, f["tiles"] = r.random() < 0.8, []
    for kind in kinds:
        t = dict(kind=STRIDED if kind == "cols" else kind, inner=N, bias=r.random() < 0.6, act=r.choice([NONE, NONE, RELU, SIGMOID]),
                 scale=r.choice([1.0, 1.0, 0.25]), glu=0, resid=None, gate=None, xtail=False, s_i=0, s_d=1, gate_rows=0, mask=None)
        wide = 64 if r.random() < 0.3 and kind != BIAS else 128
        t["glu"] = int(wide == 64)
        if r.random() < 0.3:
            t["mask"] = r.choice([(N, 1), (1, B), (0, 1)]) if not f["tiles"] or not same_mask else f["tiles"][0]["mask"] or (N, 1)
        if kind == STRIDED:
            t["ncols"] = r.choice([wide, wide, wide - 8, 36, 32, 3])
            p, h = r.choice([(128, 32), (160, 32), (32, 32 * B * N)])
            t.update(r.choice([dict(inner=M, s_o=0, s_i=p, mask=t["mask"] and (0, 1)), dict(s_o=N * p, s_i=p), dict(s_o=p, s_i=B * p)]), s_h=h)
            if r.random() < 0.5:
                t["resid"] = r.choice(["out", "own"])
                t["xtail"] = bf16 and r.random() < 0.4
            if r.random() < 0.4:
                t.update(gate=128, gate_rows=r.choice([0, 17]), act=r.choice([NONE, SIGMOID, GATE_POS]))
        elif kind == "cols":
            t["ncols"] = r.choice([wide, 20])
            step = r.choice([1, 1, 1, 2])
            cs = pad(step * B * np_ + 1, r.choice([1, 8]))
            t.update(s_o=step * np_, s_i=step, s_d=cs, s_h=32 * cs)
        elif kind == BIAS:
            t.update(ncols=r.randint(1, 8), s_o=pad(N, 32) * 32, s_h=pad(B, 32) * pad(N, 32))
        else:
            t.update(ncols=r.choice([wide, 32]), s_o=4 * pad(N, 32) * 32, s_h=pad(N, 32) * 32)
        f["tiles"].append(t)
    return f


@pytest.mark.parametrize("seed", range(8))
@pytest.mark.parametrize("chan", [False, True])
@pytest.mark.parametrize("K", [64, 96, 128, 256])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_forms_of_a_launch(dev, dtype, K, chan, seed):
    from fastfold_amd import _lib
    r = random.Random("%s %d %d %d" % (dtype, K, chan, seed))
    for _ in range(6):
        f = _form(r, dtype == torch.bfloat16, K, chan)
        g = torch.Generator().manual_seed(r.randrange(1 << 30))

        def rnd(*s):
            return torch.randn(*s, generator=g).to(dtype)
        f64 = lambda t: t.double().numpy()
        nt = lambda p, q: (torch.from_numpy(p).to(dev) @ torch.from_numpy(q).to(dev).t()).cpu().numpy()
        M, m = f["M"], np.arange(f["M"])
        a_off = ((m // f["a_inner"]) * f["a_so"] + (m % f["a_inner"]) * f["a_si"])[:, None] + np.arange(K)[None, :] * (f["a_cs"] if chan else 1)
        a, w, b, ln = rnd(int(a_off.max()) + 17), rnd(len(f["tiles"]) * 128, K) / K ** 0.5, rnd(len(f["tiles"]) * 128), (1 + 0.1 * rnd(K), 0.1 * rnd(K))
        x = f64(a)[a_off]
        if f["ln"]:
            x = ops_np.layer_norm(x, f64(ln[0]), f64(ln[1]))
            x = f64(torch.from_numpy(x).to(dtype)) if dtype == torch.bfloat16 else x
        keep, tiles, want = [], [], []

        def on_gpu(t):
            keep.append(t.to(dev))
            return keep[-1]
        mask = (torch.rand(M + 1024, generator=g) > 0.3).to(dtype)
        mask_d, b_d = on_gpu(mask), on_gpu(b)
        for i, t in enumerate(f["tiles"]):
            off = _offsets(t, M)
            init = rnd((int(off.max()) + 1 + 2047) // 1024 * 1024)          # whole operand tiles and room behind them
            ii = i * 128 + np.arange(t["ncols"])
            if t["glu"]:
                c = np.arange(t["ncols"])
                ii = i * 128 + (c >> 5) * 64 + (c & 31)
            bias = f64(b) if t["bias"] else np.zeros(len(b))
            y = nt(x, f64(w)[ii]) + bias[ii]
            if t["glu"]:
                y = y / (1 + np.exp(-(nt(x, f64(w)[ii + 32]) + bias[ii + 32])))
            elif t["act"] == RELU:
                y = np.maximum(y, 0)
            elif t["act"] == SIGMOID:
                y = 1 / (1 + np.exp(-y))
            y = y * t["scale"]
            kw = {k: t[k] for k in ("kind", "inner", "s_o", "s_i", "s_h", "s_d", "act", "ncols", "glu", "scale", "gate_rows")}
            if t["mask"]:
                y = y * f64(mask)[(m // t["inner"]) * t["mask"][0] + (m % t["inner"]) * t["mask"][1]][:, None]
                kw.update(rowmask=mask_d, m_so=t["mask"][0], m_si=t["mask"][1])
            if t["gate"]:
                gate = rnd(M if not t["gate_rows"] else t["gate_rows"], t["gate"])
                gm = f64(gate)[m % len(gate)][:, :t["ncols"]]
                y = y * ((gm > 0) if t["act"] == GATE_POS else gm)
                kw.update(gate=on_gpu(gate), gate_ld=t["gate"])
            tail = torch.zeros(len(init), dtype=torch.int8)
            if t["xtail"]:
                init[init == 0] = 1.0                                       # (0, negative tail) is no value
                tail = torch.randint(-128, 128, (len(init),), generator=g).to(torch.int8)
            pair = lambda h, u: f64(((h.view(torch.int16).int() << 16) + (u.int() << 8)).view(torch.float32)) if t["xtail"] else f64(h)
            out, tail_d = on_gpu(init), on_gpu(tail)
            src = init
            if t["resid"]:
                if t["resid"] == "own":
                    src = rnd(len(init))
                    src[src == 0] = 1.0
                y = y + pair(src, tail)[off]
                kw.update(resid=out if t["resid"] == "out" else on_gpu(src))
            ref = pair(init, tail)
            ref[off] = y
            touched = np.zeros(len(init), dtype=bool)
            touched[off] = True
            assert touched.sum() == off.size
            want.append((out, tail_d, pair, ref, touched, init))
            tiles.append(_lib.make_tile(out, bias=b_d[i * 128:] if t["bias"] else None, xtail=tail_d if t["xtail"] else None, **kw))
        what = "%s %r" % (dtype, f)
        print(what, flush=True)
        akw = dict(a_inner=f["a_inner"], a_so=f["a_so"], a_si=f["a_si"])
        if chan:
            akw.update(a_chanmajor=True, a_cs=f["a_cs"])
        _lib.fused_linear(on_gpu(a), on_gpu(w), tiles, M=M, K=K, ln=tuple(on_gpu(t) for t in ln) if f["ln"] else None, **akw)
        for i, (out, tail_d, pair, ref, touched, init) in enumerate(want):
            got = pair(out.cpu(), tail_d.cpu())
            assert np.array_equal(out.cpu().double().numpy()[~touched], init.double().numpy()[~touched]), (i, what)
            assert np.abs(got - ref)[touched].max() <= TOL[dtype] * max(1.0, np.abs(ref[touched]).max()), (i, what)
