"""GPU parity of ffk_fused_linear (through the C ABI) against float64 numpy linear algebra
(oracle.ops_np): every prologue / epilogue / layout the Evoformer modules use."""
import numpy as np
import pytest
import torch

from oracle import ops_np

pytestmark = pytest.mark.gpu

TOL = {torch.float32: 2e-5, torch.bfloat16: 2e-2}   # relative to max |ref|


def _np(t):
    return t.detach().float().cpu().numpy().astype(np.float64)


def _pack(w, n_tiles):
    out = torch.zeros(n_tiles * 128, w.shape[1], dtype=w.dtype, device=w.device)
    out[: w.shape[0]] = w
    return out


def _rel(got, ref):
    return np.abs(got - ref).max() / max(np.abs(ref).max(), 1e-6)


def _sig(x):
    return 1.0 / (1.0 + np.exp(-x))


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("M,K,N", [(300, 128, 256), (129, 256, 200), (64, 64, 36), (1000, 256, 1024)])
def test_plain_bias_relu_rowmajor(dev, dtype, M, K, N):
    from fastfold_amd import _lib
    g = torch.Generator().manual_seed(M + K)
    a = torch.randn(M, K, generator=g).to(dev, dtype)
    w = (torch.randn(N, K, generator=g) / K ** 0.5).to(dev, dtype)
    b = torch.randn(N, generator=g).to(dev, dtype)
    nt = (N + 127) // 128
    wp, bp = _pack(w, nt), torch.zeros(nt * 128, dtype=dtype, device=dev)
    bp[:N] = b
    out = torch.full((M, N), 7.0, dtype=dtype, device=dev)
    tiles = [_lib.make_tile(out.data_ptr() + i * 128 * out.element_size(), bias=bp.data_ptr() + i * 128 * out.element_size(),
                            inner=M, s_i=N, act=_lib.FFK_ACT_RELU, ncols=min(128, N - i * 128)) for i in range(nt)]
    if N % (16 // out.element_size()) != 0:
        pytest.skip("row pitch not 16-byte aligned")
    _lib.fused_linear(a, wp, tiles, M=M, K=K)
    ref = np.maximum(ops_np.linear(_np(a), _np(w), _np(b)), 0)
    assert _rel(_np(out), ref) < TOL[dtype]


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("K", [128, 256])
def test_layernorm_prologue_resid_gate_inplace(dev, dtype, K):
    from fastfold_amd import _lib
    M, N = 333, 128
    g = torch.Generator().manual_seed(K)
    a = (torch.randn(M, K, generator=g) * 2 + 0.5).to(dev, dtype)
    w = (torch.randn(N, K, generator=g) / K ** 0.5).to(dev, dtype)
    b = torch.randn(N, generator=g).to(dev, dtype)
    gam = (1 + 0.1 * torch.randn(K, generator=g)).to(dev, dtype)
    bet = (0.1 * torch.randn(K, generator=g)).to(dev, dtype)
    gate = torch.rand(M, N, generator=g).to(dev, dtype)
    z = torch.randn(M, N, generator=g).to(dev, dtype)
    z0 = z.clone()
    tiles = [_lib.make_tile(z, bias=b, resid=z, gate=gate, gate_ld=N, inner=M, s_i=N)]
    _lib.fused_linear(a, _pack(w, 1), tiles, M=M, K=K, ln=(gam, bet))
    x = ops_np.layer_norm(_np(a), _np(gam), _np(bet))
    if dtype == torch.bfloat16:
        x = _np(torch.from_numpy(x).to(torch.bfloat16))       # the kernel rounds LN output to the operand dtype
    ref = _np(z0) + _np(gate) * ops_np.linear(x, _np(w), _np(b))
    assert _rel(_np(z), ref) < TOL[dtype]


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_transposed_rows_in_and_out(dev, dtype):
    """A is z[I,J,C] traversed as (j, i); the update is written back to z[i, j]."""
    from fastfold_amd import _lib
    I, J, C = 21, 13, 128
    g = torch.Generator().manual_seed(3)
    z = torch.randn(I, J, C, generator=g).to(dev, dtype)
    w = (torch.randn(C, C, generator=g) / C ** 0.5).to(dev, dtype)
    z0 = z.clone()
    # logical row m = j * I + i  ->  z[i, j]
    tiles = [_lib.make_tile(z, resid=z, inner=I, s_o=C, s_i=J * C)]
    _lib.fused_linear(z0, _pack(w, 1), tiles, M=I * J, K=C, a_inner=I, a_so=C, a_si=J * C)
    ref = _np(z0) + ops_np.linear(_np(z0), _np(w))
    assert _rel(_np(z), ref) < TOL[dtype]


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("r", [24, 37])
def test_glu_rowmask_channel_major(dev, dtype, r):
    """Triangle-multiplication projection: (Wp x + bp) * sigmoid(Wg x + bg) * mask, stored [c][i][kpad]."""
    from fastfold_amd import _lib
    C, Ch = 128, 128
    kpad = (r + 7) // 8 * 8
    g = torch.Generator().manual_seed(r)
    z = torch.randn(r, r, C, generator=g).to(dev, dtype)
    wp = (torch.randn(Ch, C, generator=g) / C ** 0.5).to(dev, dtype)
    wg = (torch.randn(Ch, C, generator=g) / C ** 0.5).to(dev, dtype)
    bp, bg = torch.randn(Ch, generator=g).to(dev, dtype), torch.randn(Ch, generator=g).to(dev, dtype)
    mask = (torch.rand(r, r, generator=g) > 0.2).to(dev, dtype)
    # packed tiles: [p 0..31 | g 0..31 | p 32..63 | g 32..63] per 128 rows
    idx = []
    wcat, bcat = [], []
    for t in range(Ch // 64):
        for q in range(2):
            sl = slice(t * 64 + q * 32, t * 64 + q * 32 + 32)
            wcat += [wp[sl], wg[sl]]
            bcat += [bp[sl], bg[sl]]
    wpk, bpk = torch.cat(wcat).contiguous(), torch.cat(bcat).contiguous()
    for transposed in (False, True):
        out = torch.zeros(Ch, r, kpad, dtype=dtype, device=dev)
        es = out.element_size()
        tiles = []
        for t in range(Ch // 64):
            tiles.append(_lib.make_tile(out.data_ptr() + t * 64 * r * kpad * es, bias=bpk.data_ptr() + t * 128 * es,
                                        glu=1, ncols=64, inner=r, s_o=kpad, s_i=1, s_h=32 * r * kpad, s_d=r * kpad,
                                        rowmask=mask, m_so=(1 if transposed else r), m_si=(r if transposed else 1)))
        if transposed:   # logical row (a, b) reads z[b, a]
            _lib.fused_linear(z, wpk, tiles, M=r * r, K=C, a_inner=r, a_so=C, a_si=r * C)
        else:
            _lib.fused_linear(z, wpk, tiles, M=r * r, K=C)
        zz = _np(z).transpose(1, 0, 2) if transposed else _np(z)
        mm = _np(mask).T if transposed else _np(mask)
        ref = ops_np.linear(zz, _np(wp), _np(bp)) * _sig(ops_np.linear(zz, _np(wg), _np(bg))) * mm[..., None]
        got = _np(out)[:, :, :r].transpose(1, 2, 0)
        assert _rel(got, ref) < TOL[dtype]
        assert float(out[:, :, r:].abs().max()) == 0.0 if kpad > r else True


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("B2,N,H", [(3, 70, 4), (2, 32, 8)])
def test_attention_operand_tiles(dev, dtype, B2, N, H):
    from fastfold_amd import _lib
    from fastfold_amd.model.fastnn.kernel import layouts
    C = H * 32
    K = 128
    g = torch.Generator().manual_seed(N)
    x = torch.randn(B2, N, K, generator=g).to(dev, dtype)
    wq, wk, wv = ((torch.randn(C, K, generator=g) / K ** 0.5).to(dev, dtype) for _ in range(3))
    NT = layouts.n_tiles(N)
    q = torch.zeros(B2, H, NT, 2, 32, 16, dtype=dtype, device=dev)
    k = torch.zeros_like(q)
    v = torch.zeros(B2, H, NT, 2, 32, 4, 4, dtype=dtype, device=dev)
    es = q.element_size()
    tiles, ws = [], []
    for buf, w, kind, scale in ((q, wq, _lib.FFK_TILE_QK, 0.25), (k, wk, _lib.FFK_TILE_QK, 1.0), (v, wv, _lib.FFK_TILE_V, 1.0)):
        for t in range(C // 128):
            tiles.append(_lib.make_tile(buf.data_ptr() + t * 4 * NT * 1024 * es, kind=kind, inner=N, s_o=H * NT * 1024,
                                        s_h=NT * 1024, scale=scale))
            ws.append(w[t * 128:(t + 1) * 128])
    _lib.fused_linear(x, torch.cat(ws).contiguous(), tiles, M=B2 * N, K=K)
    for buf, w, un, scale in ((q, wq, layouts.untile_qk, 0.25), (k, wk, layouts.untile_qk, 1.0), (v, wv, layouts.untile_v, 1.0)):
        ref = (ops_np.linear(_np(x), _np(w)) * scale).reshape(B2, N, H, 32).transpose(0, 2, 1, 3)
        assert _rel(_np(un(buf, N)), ref) < TOL[dtype]


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("r,H", [(45, 4), (64, 8)])
def test_bias_tiles(dev, dtype, r, H):
    from fastfold_amd import _lib
    from fastfold_amd.model.fastnn.kernel import layouts
    C = 128
    g = torch.Generator().manual_seed(r)
    z = torch.randn(r, r, C, generator=g).to(dev, dtype)
    wb = (torch.randn(H, C, generator=g) / C ** 0.5).to(dev, dtype)
    gam = (1 + 0.1 * torch.randn(C, generator=g)).to(dev, dtype)
    bet = (0.1 * torch.randn(C, generator=g)).to(dev, dtype)
    T = layouts.n_tiles(r)
    for transposed in (False, True):
        bt = torch.zeros(H, T, T, 2, 32, 16, dtype=dtype, device=dev)
        tile = _lib.make_tile(bt, kind=_lib.FFK_TILE_BIAS, inner=r, s_o=T * 1024, s_h=T * T * 1024, ncols=H, scale=_lib.LOG2E)
        kw = dict(a_inner=r, a_so=C, a_si=r * C) if transposed else {}
        _lib.fused_linear(z, _pack(wb, 1), [tile], M=r * r, K=C, ln=(gam, bet), **kw)
        zz = _np(z).transpose(1, 0, 2) if transposed else _np(z)
        x = ops_np.layer_norm(zz, _np(gam), _np(bet))
        if dtype == torch.bfloat16:
            x = _np(torch.from_numpy(x).to(torch.bfloat16))
        ref = (ops_np.linear(x, _np(wb)) * _lib.LOG2E).transpose(2, 0, 1)       # [h, q, k]
        assert _rel(_np(layouts.untile_bias(bt, r, r)), ref) < TOL[dtype]


@pytest.mark.parametrize("r,H", [(45, 4), (64, 3), (33, 1)])
def test_bias_tile_rides_on_a_projection_launch(dev, r, H):
    """A trailing FFK_TILE_BIAS tile in a launch of the weights-in-registers kernel (bf16, K = 128, <= 4 heads): computed
    by small products on the slab rows, no weight slot.  Checked against numpy, against the staged kernels on the
    same descriptor, in both traversal orders; the other tile of the launch is unaffected and the padding of ragged
    bias tiles stays zero."""
    from fastfold_amd import _lib
    from fastfold_amd.model.fastnn.kernel import layouts
    dtype, C = torch.bfloat16, 128
    g = torch.Generator().manual_seed(r * 7 + H)
    z = (torch.randn(r, r, C, generator=g) * 1.3 + 0.2).to(dev, dtype)
    w = (torch.randn(128, C, generator=g) / C ** 0.5).to(dev, dtype)
    wb = (torch.randn(H, C, generator=g) / C ** 0.5).to(dev, dtype)
    gam = (1 + 0.1 * torch.randn(C, generator=g)).to(dev, dtype)
    bet = (0.1 * torch.randn(C, generator=g)).to(dev, dtype)
    wpk = torch.cat([_pack(w, 1), _pack(wb, 1)]).contiguous()
    T = layouts.n_tiles(r)
    for transposed in (False, True):
        res = []
        for staged in (False, True):
            y = torch.zeros(r * r, 128, dtype=dtype, device=dev)
            bt = torch.zeros(H, T, T, 2, 32, 16, dtype=dtype, device=dev)
            tiles = [_lib.make_tile(y, inner=r * r, s_i=128),
                     _lib.make_tile(bt, kind=_lib.FFK_TILE_BIAS, inner=r, s_o=T * 1024, s_h=T * T * 1024, ncols=H,
                                    scale=_lib.LOG2E)]
            kw = dict(a_inner=r, a_so=C, a_si=r * C) if transposed else {}
            _lib.fused_linear(z, wpk, tiles, M=r * r, K=C, ln=(gam, bet), staged=staged, **kw)
            res.append((y, bt))
        zz = _np(z).transpose(1, 0, 2) if transposed else _np(z)
        x = _np(torch.from_numpy(ops_np.layer_norm(zz, _np(gam), _np(bet))).to(dtype))
        ref = (ops_np.linear(x, _np(wb)) * _lib.LOG2E).transpose(2, 0, 1)       # [h, q, k]
        for y, bt in res:
            assert _rel(_np(layouts.untile_bias(bt, r, r)), ref) < 1e-2
            assert _rel(_np(y), ops_np.linear(x, _np(w)).reshape(r * r, 128)) < TOL[dtype]
            full = _np(layouts.untile_bias(bt, T * 32, T * 32))
            assert np.abs(full[:, r:, :]).max(initial=0.0) == 0.0 and np.abs(full[:, :, r:]).max(initial=0.0) == 0.0
        assert _rel(_np(res[0][1]), _np(res[1][1])) < 1e-2
        assert torch.equal(res[0][0], res[1][0]) or _rel(_np(res[0][0]), _np(res[1][0])) < 1e-2


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("C,with_ln", [(128, True), (64, True), (64, False)])
@pytest.mark.parametrize("r", [40, 27, 104])
def test_channel_major_a_with_layernorm(dev, dtype, r, C, with_ln):
    """Triangle-multiplication output stage: A[(i,j), c] = P[c][i][jpad], at the Evoformer's 128 channels and the
    template stack's 64."""
    from fastfold_amd import _lib
    jpad = (r + 7) // 8 * 8
    g = torch.Generator().manual_seed(r + C)
    P = torch.randn(C, r, jpad, generator=g).to(dev, dtype)
    w = (torch.randn(C, C, generator=g) / C ** 0.5).to(dev, dtype)
    gam = (1 + 0.1 * torch.randn(C, generator=g)).to(dev, dtype)
    bet = (0.1 * torch.randn(C, generator=g)).to(dev, dtype)
    b = torch.randn(C, generator=g).to(dev, dtype)
    gate = torch.rand(r * r, C, generator=g).to(dev, dtype)
    z = torch.randn(r, r, C, generator=g).to(dev, dtype)
    z0 = z.clone()
    tiles = [_lib.make_tile(z, bias=b, resid=z, gate=gate, gate_ld=C, inner=r * r, s_i=C, ncols=C)]
    _lib.fused_linear(P, _pack(w, 1), tiles, M=r * r, K=C, a_inner=r, a_so=jpad, a_si=1, a_chanmajor=True,
                      a_cs=r * jpad, ln=(gam, bet) if with_ln else None)
    x = _np(P)[:, :, :r].transpose(1, 2, 0)
    if with_ln:
        x = ops_np.layer_norm(x, _np(gam), _np(bet))
        if dtype == torch.bfloat16:
            x = _np(torch.from_numpy(x).to(torch.bfloat16))
    ref = _np(z0) + _np(gate).reshape(r, r, C) * ops_np.linear(x, _np(w), _np(b))
    assert _rel(_np(z), ref) < TOL[dtype]


def test_bad_descriptors_are_rejected(dev):
    from fastfold_amd import _lib
    a = torch.zeros(64, 100, device=dev)
    w = torch.zeros(128, 100, device=dev)
    out = torch.zeros(64, 128, device=dev)
    with pytest.raises(RuntimeError):
        _lib.fused_linear(a, w, [_lib.make_tile(out, inner=64, s_i=128)], M=64, K=100)     # K % 32
    a = torch.zeros(64, 128, device=dev)
    w = torch.zeros(128, 128, device=dev)
    with pytest.raises(RuntimeError):
        _lib.fused_linear(a, w, [_lib.make_tile(out, inner=0, s_i=128)], M=64, K=128)      # inner
    with pytest.raises(RuntimeError):
        _lib.fused_linear(a, w, [_lib.make_tile(out, inner=64, s_i=128, s_d=2, resid=out)], M=64, K=128)


def test_weights_stationary_many_slabs(dev):
    """bf16, K = 128, more slabs than workgroups (persistent loop, ragged last slab): q in accumulator
    order with a scale, k in q/k order, v, a sigmoid gate in accumulator order and a plain relu tile,
    all from one LayerNorm-ed pass over A."""
    from fastfold_amd import _lib
    from fastfold_amd.model.fastnn.kernel import layouts
    dtype = torch.bfloat16
    B2, N, H, K = 131, 288, 4, 128                      # M = 37728 rows = 294.75 slabs
    C = H * 32
    M = B2 * N
    g = torch.Generator().manual_seed(11)
    x = (torch.randn(B2, N, K, generator=g) + 0.3).to(dev, dtype)
    ws_ = [(torch.randn(C, K, generator=g) / K ** 0.5).to(dev, dtype) for _ in range(5)]
    bias_g = torch.randn(C, generator=g).to(dev, dtype)
    bias_r = torch.randn(C, generator=g).to(dev, dtype)
    gam = (1 + 0.1 * torch.randn(K, generator=g)).to(dev, dtype)
    bet = (0.1 * torch.randn(K, generator=g)).to(dev, dtype)
    NT = layouts.n_tiles(N)
    q = torch.zeros(B2, H, NT, 2, 32, 4, 4, dtype=dtype, device=dev)
    k = torch.zeros(B2, H, NT, 2, 32, 16, dtype=dtype, device=dev)
    v = torch.zeros(B2, H, NT, 2, 32, 4, 4, dtype=dtype, device=dev)
    gt = torch.zeros(B2, H, NT, 2, 32, 4, 4, dtype=dtype, device=dev)
    plain = torch.zeros(M, C, dtype=dtype, device=dev)
    tk = dict(inner=N, s_o=H * NT * 1024, s_h=NT * 1024)
    tiles = [_lib.make_tile(q, kind=_lib.FFK_TILE_ACC, scale=0.25, **tk),
             _lib.make_tile(k, kind=_lib.FFK_TILE_QK, **tk),
             _lib.make_tile(v, kind=_lib.FFK_TILE_V, **tk),
             _lib.make_tile(gt, kind=_lib.FFK_TILE_ACC, bias=bias_g, act=_lib.FFK_ACT_SIGMOID, **tk),
             _lib.make_tile(plain, bias=bias_r, act=_lib.FFK_ACT_RELU, inner=M, s_i=C)]
    bias_all = torch.zeros(5 * 128, dtype=dtype, device=dev)
    bias_all[3 * 128:4 * 128] = bias_g
    bias_all[4 * 128:] = bias_r
    tiles[3].bias = bias_all.data_ptr() + 3 * 128 * 2
    tiles[4].bias = bias_all.data_ptr() + 4 * 128 * 2
    _lib.fused_linear(x, torch.cat(ws_).contiguous(), tiles, M=M, K=K, ln=(gam, bet))
    xn = _np(torch.from_numpy(ops_np.layer_norm(_np(x), _np(gam), _np(bet))).to(torch.bfloat16))
    lin = [ops_np.linear(xn, _np(w)) for w in ws_]
    heads = lambda y: y.reshape(B2, N, H, 32).transpose(0, 2, 1, 3)
    assert _rel(_np(layouts.untile_rows_acc(q, N)), heads(lin[0] * 0.25)) < TOL[dtype]
    assert _rel(_np(layouts.untile_qk(k, N)), heads(lin[1])) < TOL[dtype]
    assert _rel(_np(layouts.untile_v(v, N)), heads(lin[2])) < TOL[dtype]
    assert _rel(_np(layouts.untile_rows_acc(gt, N)), heads(_sig(lin[3] + _np(bias_g)))) < TOL[dtype]
    assert _rel(_np(plain).reshape(B2, N, C), np.maximum(lin[4] + _np(bias_r), 0)) < TOL[dtype]


def test_weights_stationary_matches_other_variant(dev):
    """GLU + row mask, channel-major store, both traversal orders, at a multi-slab size: the
    weights-stationary kernel and the LDS-staged kernel must agree to bf16 rounding."""
    from fastfold_amd import _lib
    dtype = torch.bfloat16
    r, C, Ch = 200, 128, 128
    g = torch.Generator().manual_seed(5)
    z = torch.randn(r, r, C, generator=g).to(dev, dtype)
    wpk = (torch.randn(2 * Ch + 128, C, generator=g) / C ** 0.5).to(dev, dtype)
    bpk = torch.randn(2 * Ch + 128, generator=g).to(dev, dtype)
    gam = (1 + 0.1 * torch.randn(C, generator=g)).to(dev, dtype)
    bet = (0.1 * torch.randn(C, generator=g)).to(dev, dtype)
    mask = (torch.rand(r, r, generator=g) > 0.2).to(dev, dtype)
    outs = []
    for no_ws in (False, True):
        res = []
        for transposed in (False, True):
            out = torch.zeros(Ch, r, r, dtype=dtype, device=dev)
            gate = torch.zeros(r * r, C, dtype=dtype, device=dev)
            tiles = []
            for t in range(Ch // 64):
                tiles.append(_lib.make_tile(out.data_ptr() + t * 64 * r * r * 2, bias=bpk.data_ptr() + t * 128 * 2,
                                            glu=1, ncols=64, inner=r, s_o=r, s_i=1, s_h=32 * r * r, s_d=r * r,
                                            rowmask=mask, m_so=(1 if transposed else r), m_si=(r if transposed else 1)))
            kw = dict(inner=r, s_o=C, s_i=r * C) if transposed else dict(inner=r * r, s_i=C)
            tiles.append(_lib.make_tile(gate, bias=bpk.data_ptr() + 2 * 128 * 2, act=_lib.FFK_ACT_SIGMOID, **kw))
            akw = dict(a_inner=r, a_so=C, a_si=r * C) if transposed else {}
            _lib.fused_linear(z, wpk, tiles, M=r * r, K=C, ln=(gam, bet), staged=no_ws, **akw)
            res += [out, gate]
        outs.append(res)
    for a, b in zip(*outs):
        assert float(a.float().abs().max()) > 0.1
        assert _rel(_np(a), _np(b)) < 1e-2


@pytest.mark.parametrize("r,H,C", [(45, 4, 128), (64, 8, 128), (96, 4, 128), (45, 4, 64), (64, 4, 64)])
def test_pair_bias_kernel(dev, r, H, C):
    """ffk_pair_bias (bf16): LayerNorm + H-row projection written as attention bias tiles, in both
    traversal orders, against float64 numpy."""
    from fastfold_amd import _lib
    from fastfold_amd.model.fastnn.kernel import layouts
    dtype = torch.bfloat16
    g = torch.Generator().manual_seed(r + H)
    z = (torch.randn(r, r, C, generator=g) * 1.5 + 0.4).to(dev, dtype)
    wb = (torch.randn(H, C, generator=g) / C ** 0.5).to(dev, dtype)
    gam = (1 + 0.1 * torch.randn(C, generator=g)).to(dev, dtype)
    bet = (0.1 * torch.randn(C, generator=g)).to(dev, dtype)
    T = layouts.n_tiles(r)
    scratch = torch.empty(16 * C + 16, dtype=torch.float32, device=dev)
    for transposed in (False, True):
        bt = torch.zeros(H, T, T, 2, 32, 16, dtype=dtype, device=dev)
        kw = dict(a_inner=r, a_so=C, a_si=r * C) if transposed else dict(a_inner=r * r, a_so=0, a_si=C)
        _lib.pair_bias(bt, z, gam, bet, wb, scratch, N=r, C=C, H=H, scale=_lib.LOG2E, **kw)
        zz = _np(z).transpose(1, 0, 2) if transposed else _np(z)
        x = ops_np.layer_norm(zz, _np(gam), _np(bet))
        ref = (ops_np.linear(x, _np(wb)) * _lib.LOG2E).transpose(2, 0, 1)       # [h, q, k]
        assert _rel(_np(layouts.untile_bias(bt, r, r)), ref) < TOL[dtype]
        # a later call may reuse the weight operand the first one left in scratch (w = None)
        bt2 = torch.zeros_like(bt)
        _lib.pair_bias(bt2, z, None, None, None, scratch, N=r, C=C, H=H, scale=_lib.LOG2E, **kw)
        assert torch.equal(bt2, bt)
        # padding of ragged tiles is left untouched (zero)
        full = _np(layouts.untile_bias(bt, T * 32, T * 32))
        assert np.abs(full[:, r:, :]).max(initial=0.0) == 0.0 and np.abs(full[:, :, r:]).max(initial=0.0) == 0.0


@pytest.mark.parametrize("r,s", [(64, 128), (96, 64)])
def test_opm_fused_kernel(dev, r, s):
    """ffk_opm_fused against float64 numpy: out = resid + (sum_{d,e} (a_i^T b_j)[d,e] W[c,d,e] + bias) / (norm + eps)."""
    from fastfold_amd import _lib
    dtype = torch.bfloat16
    g = torch.Generator().manual_seed(r + s)
    a_t = (torch.randn(r * 32, s, generator=g) * 0.5).to(dev, dtype)       # row i*32 + d, K = sequences
    b_t = (torch.randn(r * 32, s, generator=g) * 0.5).to(dev, dtype)
    w = (torch.randn(128, 32, 32, generator=g) / 32).to(dev, dtype)         # [c, d, e] as in the reference weight
    bias = torch.randn(128, generator=g).to(dev, dtype)
    norm = (torch.rand(r, r, generator=g) * s + 1).to(dev)
    resid = torch.randn(r * r, 128, generator=g).to(dev, dtype)
    out = torch.empty_like(resid)
    w_ed = w.transpose(1, 2).reshape(128, 1024).contiguous()
    _lib.opm_fused(out, resid, a_t, b_t, w_ed, bias, norm, r=r, spad=s, eps=1e-3)
    A = _np(a_t).reshape(r, 32, s)
    B = _np(b_t).reshape(r, 32, s)
    O = np.einsum("ids,jes->ijde", A, B)
    O = _np(torch.from_numpy(O).to(torch.bfloat16))                         # the kernel rounds the outer product to bf16
    upd = (np.einsum("ijde,cde->ijc", O, _np(w)) + _np(bias)) / (_np(norm)[..., None] + 1e-3)
    got = _np(out).reshape(r, r, 128) - _np(resid).reshape(r, r, 128)
    assert _rel(got, upd) < TOL[dtype]
    # in place
    res2 = resid.clone()
    _lib.opm_fused(res2, res2, a_t, b_t, w_ed, bias, norm, r=r, spad=s, eps=1e-3)
    assert torch.equal(res2, out)
    with pytest.raises(RuntimeError):
        _lib.opm_fused(out, resid, a_t, b_t, w_ed, bias, norm, r=r + 8, spad=s, eps=1e-3)


@pytest.mark.parametrize("C", [128, 256])
@pytest.mark.parametrize("M", [256, 1000, 70000])
def test_transition_fused_kernel(dev, M, C):
    """ffk_transition_fused (pair width 128, MSA width 256) against float64 numpy, including a ragged last workgroup
    and in-place use."""
    from fastfold_amd import _lib
    dtype = torch.bfloat16
    Hd = 4 * C
    g = torch.Generator().manual_seed(M + C)
    x = (torch.randn(M, C, generator=g) * 1.5 + 0.2).to(dev, dtype)
    gam = (1 + 0.1 * torch.randn(C, generator=g)).to(dev, dtype)
    bet = (0.1 * torch.randn(C, generator=g)).to(dev, dtype)
    w1 = (torch.randn(Hd, C, generator=g) / C ** 0.5).to(dev, dtype)
    b1 = torch.randn(Hd, generator=g).to(dev, dtype)
    w2 = (torch.randn(C, Hd, generator=g) / Hd ** 0.5).to(dev, dtype)
    b2 = torch.randn(C, generator=g).to(dev, dtype)
    out = torch.full_like(x, 7.0)
    _lib.transition_fused(out, x, gam, bet, w1, b1, w2, b2, M=M, C=C, hidden=Hd)
    xn = _np(torch.from_numpy(ops_np.layer_norm(_np(x), _np(gam), _np(bet))).to(torch.bfloat16))
    h = np.maximum(ops_np.linear(xn, _np(w1), _np(b1)), 0)
    h = _np(torch.from_numpy(h).to(torch.bfloat16))                         # hidden is rounded to bf16 on chip
    upd = ops_np.linear(h, _np(w2), _np(b2))
    assert _rel(_np(out) - _np(x), upd) < TOL[dtype]
    x2 = x.clone()
    _lib.transition_fused(x2, x2, gam, bet, w1, b1, w2, b2, M=M, C=C, hidden=Hd)
    assert torch.equal(x2, out)
    with pytest.raises(RuntimeError):
        _lib.transition_fused(out, x, gam, bet, w1, b1, w2, b2, M=M, C=64, hidden=256)
    with pytest.raises(RuntimeError):
        _lib.transition_fused(out, x, gam, bet, w1, b1, w2, b2, M=M, C=C, hidden=2 * C)


@pytest.mark.parametrize("r", [64, 104])
def test_fused_linear_second_operand(dev, r):
    """GLU tiles whose gate halves come from a second operand (the output stage of the triangle multiplication):
    out = resid + (W_p LN2(p) + b_p) * sigmoid(W_g LN1(z) + b_g), p channel-major, both LayerNorms folded into
    the packed weights (statistics taken from the operand fragments inside the kernel)."""
    from fastfold_amd import _lib
    from fastfold_amd.model.fastnn import _fused as F_
    dtype = torch.bfloat16
    C, M = 128, r * r
    g = torch.Generator().manual_seed(r)
    p_cm = (torch.randn(C, r, r, generator=g) * 2 + 0.3).to(dev, dtype)            # [c, i, j]
    z = (torch.randn(M, C, generator=g) * 1.5 - 0.2).to(dev, dtype)
    gam1, gam2 = ((1 + 0.1 * torch.randn(C, generator=g)).to(dev, dtype) for _ in range(2))
    bet1, bet2 = ((0.1 * torch.randn(C, generator=g)).to(dev, dtype) for _ in range(2))
    wp, wg = ((torch.randn(C, C, generator=g) / C ** 0.5).to(dev, dtype) for _ in range(2))
    bp, bg = (torch.randn(C, generator=g).to(dev, dtype) for _ in range(2))
    w_pk, b_pk, rowsums = F_.pack_trimul_out(wp, bp, wg, bg, C, dtype, dev, ln_p=(gam2, bet2), ln_z=(gam1, bet1))
    out = torch.empty(M, C, device=dev, dtype=dtype)
    tiles = [_lib.make_tile(out.data_ptr() + t * 64 * 2, bias=b_pk.data_ptr() + t * 128 * 2, glu=1, ncols=64,
                            resid=z.data_ptr() + t * 64 * 2, inner=M, s_i=C) for t in range(2)]
    kw = dict(M=M, K=C, a_inner=r, a_so=r, a_si=1, a_chanmajor=True, a_cs=r * r, ln_rowsums=rowsums, a2_inner=M, a2_si=C)
    _lib.fused_linear(p_cm, w_pk, tiles, a2=z, **kw)
    pn = ops_np.layer_norm(_np(p_cm).reshape(C, M).T, _np(gam2), _np(bet2))
    zn = ops_np.layer_norm(_np(z), _np(gam1), _np(bet1))
    upd = ops_np.linear(pn, _np(wp), _np(bp)) / (1 + np.exp(-ops_np.linear(zn, _np(wg), _np(bg))))
    assert _rel(_np(out) - _np(z), upd) < TOL[dtype]
    # in place on the second operand / residual
    z2 = z.clone()
    tiles = [_lib.make_tile(z2.data_ptr() + t * 64 * 2, bias=b_pk.data_ptr() + t * 128 * 2, glu=1, ncols=64,
                            resid=z2.data_ptr() + t * 64 * 2, inner=M, s_i=C) for t in range(2)]
    _lib.fused_linear(p_cm, w_pk, tiles, a2=z2, **kw)
    assert torch.equal(z2, out)
    # rows with a large common offset: the folded form subtracts mean * rowsum after the product
    p_off = (p_cm.float() + 40.0).to(dtype)
    out3 = torch.empty_like(out)
    tiles3 = [_lib.make_tile(out3.data_ptr() + t * 64 * 2, bias=b_pk.data_ptr() + t * 128 * 2, glu=1, ncols=64,
                             resid=z.data_ptr() + t * 64 * 2, inner=M, s_i=C) for t in range(2)]
    _lib.fused_linear(p_off, w_pk, tiles3, a2=z, **kw)
    pn = ops_np.layer_norm(_np(p_off).reshape(C, M).T, _np(gam2), _np(bet2))
    upd = ops_np.linear(pn, _np(wp), _np(bp)) / (1 + np.exp(-ops_np.linear(zn, _np(wg), _np(bg))))
    assert _rel(_np(out3) - _np(z), upd) < TOL[dtype]
    # a second operand without the shapes it is built for, or without folded LayerNorms, is refused, not ignored
    with pytest.raises(RuntimeError):
        _lib.fused_linear(z, w_pk, tiles, M=M, K=C, ln_rowsums=rowsums, a2=z, a2_inner=M, a2_si=C)
    with pytest.raises(RuntimeError):
        _lib.fused_linear(p_cm, w_pk, tiles, M=M, K=C, a_inner=r, a_so=r, a_si=1, a_chanmajor=True, a_cs=r * r,
                          ln=(gam2, bet2), a2=z, a2_inner=M, a2_si=C)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("K,N,P", [(64, 64, 37), (128, 128, 16)])
def test_periodic_gate_rows(dev, dtype, K, N, P):
    """gate_rows = P: logical row m is multiplied by gate row m % P (one multiplier row per column of an
    [S, P] grid of rows, as the global column attention uses it)."""
    from fastfold_amd import _lib
    S = 9
    M = S * P
    g = torch.Generator().manual_seed(K + P)
    a = torch.randn(M, K, generator=g).to(dev, dtype)
    w = (torch.randn(N, K, generator=g) / K ** 0.5).to(dev, dtype)
    b = torch.randn(N, generator=g).to(dev, dtype)
    gate = torch.randn(P, N, generator=g).to(dev, dtype)
    out = torch.empty(M, N, dtype=dtype, device=dev)
    bp = torch.zeros(128, dtype=dtype, device=dev)
    bp[:N] = b
    tiles = [_lib.make_tile(out, bias=bp, gate=gate, gate_ld=N, gate_rows=P, inner=M, s_i=N, ncols=N,
                            act=_lib.FFK_ACT_SIGMOID)]
    _lib.fused_linear(a, _pack(w, 1), tiles, M=M, K=K)
    y = 1.0 / (1.0 + np.exp(-ops_np.linear(_np(a), _np(w), _np(b))))
    ref = y.reshape(S, P, N) * _np(gate)[None]
    assert _rel(_np(out).reshape(S, P, N), ref) < TOL[dtype]


@pytest.mark.parametrize("M,nt", [(1, 3), (65, 5), (64 * 511, 2), (64 * 512, 2)])
def test_tiles_spread_over_workgroups(dev, M, nt):
    """Few rows: several workgroups share a slab, each with some of the N-tiles (also an uneven share of them)."""
    from fastfold_amd import _lib
    F = torch.nn.functional
    g = torch.Generator().manual_seed(M + nt)
    K, N = 64, 128 * nt
    x, w, b = (torch.randn(*sh, generator=g).to(dev) for sh in ((M, K), (N, K), (N,)))
    ln = (torch.rand(K, generator=g).to(dev) + 0.5, torch.randn(K, generator=g).to(dev))
    out = torch.full((M, N), float("nan"), device=dev)
    tiles = [_lib.make_tile(out.data_ptr() + 512 * i, inner=M, s_i=N, bias=b.data_ptr() + 512 * i) for i in range(nt)]
    _lib.fused_linear(x, w, tiles, M=M, K=K, ln=ln)
    ref = F.linear(F.layer_norm(x, (K,), *ln), w, b)
    torch.testing.assert_close(out, ref, rtol=1e-4, atol=2e-4)


@pytest.mark.parametrize("case", ["attention", "glu", "plain"])
def test_fp32_weights_stationary_matches_staged(dev, case):
    """Long fp32 launches: ragged last slabs, operand tiles of a row length that is no multiple of 32, channel-major GLU tiles beside
    plain ones, gate, residual and a partly filled last tile; the staged kernel normalises and multiplies in the same order."""
    from fastfold_amd import _lib
    g = torch.Generator().manual_seed(3)
    rnd = lambda *sh: torch.randn(*sh, generator=g).to(dev)
    r, K, nt = {"attention": (97, 128, 9), "glu": (176, 128, 5), "plain": (97, 256, 4)}[case]
    M = r * r
    x, w, b = rnd(M, K), rnd(nt * 128, K) / K ** 0.5, rnd(nt * 128)
    ln, mask = (rnd(K), rnd(K)), (rnd(r) > 0).float()
    gate, resid, NT = rnd(M, 512), rnd(M, 512), (r + 31) // 32
    got = []
    for staged in (True, False):
        bp = lambda i: b.data_ptr() + 512 * i
        if case == "attention":
            outs = [torch.zeros(r, 4, NT, 1024, device=dev) for _ in range(8)] + [torch.zeros(4, NT, NT, 1024, device=dev)]
            kinds = [_lib.FFK_TILE_QK, _lib.FFK_TILE_V, _lib.FFK_TILE_ACC, _lib.FFK_TILE_V] * 2
            tiles = [_lib.make_tile(o, kind=k, inner=r, s_o=4 * NT * 1024, s_h=NT * 1024, bias=bp(i), scale=0.5 + i, act=i % 3,
                                    rowmask=mask if i > 5 else None, m_si=1) for i, (o, k) in enumerate(zip(outs, kinds))]
            tiles.append(_lib.make_tile(outs[8], kind=_lib.FFK_TILE_BIAS, inner=r, s_o=NT * 1024, s_h=NT * NT * 1024, ncols=4, bias=bp(8)))
        elif case == "glu":
            outs = [torch.zeros(256, M, device=dev), torch.zeros(M, 128, device=dev)]
            tiles = [_lib.make_tile(outs[0].data_ptr() + 256 * i * M, inner=r, s_o=r, s_i=1, s_h=32 * M, s_d=M, glu=1, ncols=64,
                                    bias=bp(i), rowmask=mask, m_so=1) for i in range(4)]
            tiles.append(_lib.make_tile(outs[1], inner=M, s_i=128, bias=bp(4), act=_lib.FFK_ACT_SIGMOID))
        else:
            outs = [torch.zeros(M, 512, device=dev)]
            tiles = [_lib.make_tile(outs[0].data_ptr() + 512 * i, inner=M, s_i=512, bias=bp(i), ncols=128 if i < 3 else 36,
                                    gate=gate.data_ptr() + 512 * i if i % 2 else None, gate_ld=512,
                                    resid=resid.data_ptr() + 512 * i if i else None) for i in range(nt)]
        _lib.fused_linear(x, w, tiles, M=M, K=K, ln=ln, staged=staged)
        got.append(outs)
    for a, c in zip(*got):
        assert torch.isfinite(a).all() and float((a - c).abs().max()) <= 1e-5 * float(a.abs().max())


@pytest.mark.parametrize("K", [64, 128, 256])
@pytest.mark.parametrize("N,M", [(96, 33), (288, 129), (416, 700), (544, 1000), (1024, 130)])
def test_weights_stationary_unit_shares(dev, K, N, M):
    """Unit counts that are shared by several waves (3 of 9, 13), fill a column group (16 of 17) or two of them (32)."""
    from fastfold_amd import _lib
    F = torch.nn.functional
    g = torch.Generator().manual_seed(N + K)
    x, w, b = (torch.randn(*sh, generator=g).to(dev, torch.bfloat16) for sh in ((M, K), (N, K), (N,)))
    ln = (torch.rand(K, generator=g).to(dev, torch.bfloat16) + 0.5, torch.randn(K, generator=g).to(dev, torch.bfloat16))
    nt = (N + 127) // 128
    wp, bp = _pack(w, nt), F.pad(b, (0, nt * 128 - N))
    out = torch.full((M, N), float("nan"), dtype=torch.bfloat16, device=dev)
    tiles = [_lib.make_tile(out.data_ptr() + 256 * i, inner=M, s_i=N, bias=bp.data_ptr() + 256 * i, ncols=min(128, N - 128 * i)) for i in range(nt)]
    _lib.fused_linear(x, wp, tiles, M=M, K=K, ln=ln)
    ref = F.linear(F.layer_norm(x.float(), (K,), ln[0].float(), ln[1].float()), w.float(), b.float())
    assert torch.isfinite(out).all() and float((out.float() - ref).norm() / ref.norm()) < 6e-3


@pytest.mark.parametrize("K", [64, 128, 256])
@pytest.mark.parametrize("B2,N", [(1, 32), (3, 96), (70, 96), (300, 128), (5, 48), (9, 33), (1001, 33)])
def test_row_major_layouts(dev, K, B2, N):
    """Every epilogue of the row-major kernel from one row group to several rounds of its largest slabs, with groups that end in
    the middle of an outer step (N = 48, 33), against the LDS-staged kernels: the same products, rounded once (2^-8)."""
    from fastfold_amd import _lib
    bf = torch.bfloat16
    M, NT = B2 * N, (N + 31) // 32
    g = torch.Generator().manual_seed(K + M)

    def rnd(*s):
        return torch.randn(*s, generator=g).to(dev, bf)
    x, w, b = rnd(M, K), rnd(640, K) / K ** 0.5, rnd(640)
    ln = (1 + 0.1 * rnd(K), 0.1 * rnd(K))
    mask, gate = (torch.rand(B2, N, generator=g) > 0.2).to(dev, bf), rnd(17, 128)
    resid, tail = rnd(M, 128), torch.randint(-128, 128, (M, 128), generator=g).to(dev, torch.int8)
    resid[resid == 0] = 1.0                              # (0, negative tail) is no value: the pair would be below zero
    got = []
    for staged in (False, True):
        bp = [b.data_ptr() + 256 * i for i in range(5)]
        outs = [torch.zeros(B2, 4, NT, 1024, device=dev, dtype=bf) for _ in range(4)]
        outs += [torch.zeros(M, 256, device=dev, dtype=bf), resid.clone(), tail.clone(), torch.zeros(M, 128, device=dev, dtype=bf)]
        rows = [_lib.make_tile(outs[4].data_ptr() + 256 * i, bias=bp[i], act=_lib.FFK_ACT_RELU, inner=M, s_i=256, ncols=(128, 104)[i]) for i in range(2)]
        if N % 32 == 0:
            tk = dict(inner=N, s_o=4 * NT * 1024, s_h=NT * 1024)
            rows += [_lib.make_tile(outs[0], kind=_lib.FFK_TILE_V, **tk), _lib.make_tile(outs[1], kind=_lib.FFK_TILE_QK, scale=0.25, **tk),
                     _lib.make_tile(outs[2], kind=_lib.FFK_TILE_ACC, bias=bp[4], act=_lib.FFK_ACT_SIGMOID, **tk)]
        _lib.fused_linear(x, w, rows, M=M, K=K, a_inner=N, a_so=N * K, a_si=K, ln=ln, staged=staged)
        # residual with a tail in place, rows of the tensor taken column by column, a multiplier shared by every 17th row
        _lib.fused_linear(x, w, [_lib.make_tile(outs[5], bias=bp[0], resid=outs[5], xtail=outs[6], gate=gate, gate_ld=128, gate_rows=17,
                                                inner=N, s_o=128, s_i=B2 * 128)], M=M, K=K, staged=staged)
        _lib.fused_linear(x, w, [_lib.make_tile(outs[7], resid=resid, inner=N, s_o=128, s_i=B2 * 128, ncols=72)], M=M, K=K, staged=staged)
        if N % 16 == 0 and M % 16 == 0 and K != 256:
            cm = torch.zeros(64, B2 * N + 16, device=dev, dtype=bf)
            _lib.fused_linear(x, w, [_lib.make_tile(cm, glu=1, ncols=64, bias=bp[1], inner=N, s_o=N, s_i=1, s_h=32 * cm.shape[1], s_d=cm.shape[1],
                                                    rowmask=mask, m_so=N, m_si=1)], M=M, K=K, ln=ln, staged=staged)
            outs.append(cm)
        got.append(outs)
    got[0][6], got[1][6] = [((o[5].view(torch.int16).int() << 16) + (o[6].int() << 8)).view(torch.float32) for o in got]    # 24-bit values
    for i, (a, c) in enumerate(zip(*got)):
        assert torch.isfinite(a.float()).all() and _rel(_np(a), _np(c)) < 2 ** -7, i


@pytest.mark.parametrize("K,units,M,kind", [(64, 12, 32763, "tail"), (64, 12, 32763, "resid"), (64, 20, 32763, "plain"), (128, 6, 32763, "tail"),
                                            (128, 3, 32763, "plain"), (128, 2, 9211, "glu"), (128, 12, 16379, "glu"), (256, 24, 16379, "plain")])
def test_row_major_layouts_of_many_units(dev, K, units, M, kind):
    """Launches that take the layouts of eight waves and of two units per wave, and of four waves over 64 rows, with a ragged last
    slab, against the LDS-staged kernels (the same products, rounded once)."""
    from fastfold_amd import _lib
    bf = torch.bfloat16
    g = torch.Generator(device=dev).manual_seed(K + units)

    def rnd(*s):
        return torch.randn(*s, device=dev, generator=g).to(bf)
    C = 64 if kind == "glu" else 128                  # channels per tile
    nt, N = -(-units * 32 // C), units * 32
    x, w, b, ln = rnd(M, K), rnd(nt * 128, K) / K ** 0.5, rnd(nt * 128), (1 + 0.1 * rnd(K), 0.1 * rnd(K))
    init, tail = rnd(M, nt * C), torch.randint(-128, 128, (M, nt * C), device=dev, generator=g).to(torch.int8)
    init[init == 0] = 1.0
    got = []
    for staged in (False, True):
        y, t = init.clone(), tail.clone()
        at = lambda p, i: p.data_ptr() + i * C * p.element_size()
        tiles = [_lib.make_tile(at(y, i), bias=b.data_ptr() + 256 * i, inner=M, s_i=nt * C, glu=int(kind == "glu"), ncols=min(C, N - i * C),
                                resid=at(y, i) if kind in ("resid", "tail") else None, xtail=at(t, i) if kind == "tail" else None) for i in range(nt)]
        _lib.fused_linear(x, w, tiles, M=M, K=K, ln=ln, staged=staged)
        got.append(((y.view(torch.int16).int() << 16) + (t.int() << 8)).view(torch.float32) if kind == "tail" else y)
    assert torch.isfinite(got[0].float()).all() and float((got[0].float() - got[1].float()).abs().max()) < 2 ** -7 * float(got[1].float().abs().max())


@pytest.mark.parametrize("K", [128, 256])
@pytest.mark.parametrize("B,N", [(1, 1), (3, 37), (64, 64), (131, 96), (260, 128)])
def test_fp32_row_layouts(dev, K, B, N):
    """fp32 launches from one row to both sides of the persistent layout, row groups that end in the middle of an outer step and
    channel-major operands and outputs of any extent, against the LDS-staged kernel (32-bit sums in another order: 1e-5)."""
    from fastfold_amd import _lib
    M = B * N
    g = torch.Generator().manual_seed(K + M)

    def rnd(*s):
        return torch.randn(*s, generator=g).to(dev)
    x, w, b = rnd(M, K), rnd(512, K) / K ** 0.5, rnd(512)
    ln = (1 + 0.1 * rnd(K), 0.1 * rnd(K))
    mask, gate, resid = (torch.rand(B, N, generator=g) > 0.2).to(dev, torch.float32), rnd(M, 128), rnd(M, 128)
    kp = (N + 3) // 4 * 4
    got = []
    for staged in (False, True):
        bp = [b.data_ptr() + 512 * i for i in range(4)]
        plain, out, cm = torch.zeros(M, 512, device=dev), torch.zeros(M, 128, device=dev), torch.zeros(64, B * kp + 16, device=dev)
        _lib.fused_linear(x, w, [_lib.make_tile(plain.data_ptr() + 512 * i, bias=bp[i], act=_lib.FFK_ACT_RELU, inner=M, s_i=512, ncols=(128, 128, 128, 36)[i])
                                 for i in range(4)], M=M, K=K, ln=ln, staged=staged)
        _lib.fused_linear(x, w, [_lib.make_tile(out, bias=bp[0], gate=gate, gate_ld=128, resid=resid, inner=N, s_o=128, s_i=B * 128)], M=M, K=K,
                          a_inner=N, a_so=N * K, a_si=K, ln=ln, staged=staged)
        outs = [plain, out]
        if K == 128:
            _lib.fused_linear(x, w, [_lib.make_tile(cm, glu=1, ncols=64, bias=bp[1], inner=N, s_o=kp, s_i=1, s_h=32 * cm.shape[1], s_d=cm.shape[1],
                                                    rowmask=mask, m_so=N, m_si=1)], M=M, K=K, ln=ln, staged=staged)
            xt = torch.zeros(K, B * kp + 4, device=dev)
            for i in range(B):
                xt[:, i * kp:i * kp + N] = x[i * N:(i + 1) * N].t()
            back = torch.zeros(M, 128, device=dev)
            _lib.fused_linear(xt, w, [_lib.make_tile(back, bias=bp[2], gate=gate, gate_ld=128, resid=resid, inner=M, s_i=128)], M=M, K=K,
                              a_inner=N, a_so=kp, a_si=1, a_chanmajor=True, a_cs=xt.shape[1], ln=ln, staged=staged)
            outs += [cm, back]
        got.append(outs)
    for i, (a, c) in enumerate(zip(*got)):
        assert torch.isfinite(a).all() and float((a - c).abs().max()) <= 1e-5 * float(c.abs().max()), i


@pytest.mark.parametrize("C", [128, 256])
def test_transition_kernels_agree(dev, C):
    """Rows of a launch get the same bits whichever kernel and workgroup size the row count selects (and so a piece of a
    tensor those of the whole), with ragged last workgroups and residual tails, in place."""
    from fastfold_amd import _lib
    g = torch.Generator().manual_seed(C)

    def rnd(*s):
        return torch.randn(*s, generator=g).to(dev, torch.bfloat16)
    M, H = 49300, 4 * C
    x, tail = rnd(M, C), torch.randint(-128, 128, (M, C), generator=g).to(dev, torch.int8)
    ln, w1, b1, w2, b2 = (1 + 0.1 * rnd(C), 0.1 * rnd(C)), rnd(H, C) / C ** 0.5, rnd(H), rnd(C, H) / H ** 0.5, rnd(C)

    def run(n):
        y, t = x[:n].clone(), tail[:n].clone()
        _lib.transition_fused(y, y, ln[0], ln[1], w1, b1, w2, b2, M=n, C=C, hidden=H, xtail=t)
        return y, t
    whole = run(M)
    h = torch.relu(torch.nn.functional.linear(torch.nn.functional.layer_norm(x.float(), (C,), ln[0].float(), ln[1].float()), w1.float(), b1.float()))
    ref = x.float() + torch.nn.functional.linear(h, w2.float(), b2.float())
    assert float((whole[0].float() - ref).norm() / ref.norm()) < 6e-3
    for n in (1, 63, 64, 65 * 64 - 5, 64 * 256, 64 * 256 + 1, 128 * 256, 128 * 256 + 1):
        y, t = run(n)
        assert torch.equal(y, whole[0][:n]) and torch.equal(t, whole[1][:n]), n


@pytest.mark.parametrize("s", [64, 128])
def test_opm_workgroup_sizes_agree(dev, s):
    """A residue pair's update has the same bits whichever number of residues per workgroup the extent selects (two up to 128, four
    at 160, eight from 192), with and without a tail."""
    from fastfold_amd import _lib
    g = torch.Generator().manual_seed(s)

    def rnd(*sh):
        return torch.randn(*sh, generator=g).to(dev, torch.bfloat16)
    R = 192
    z, ab, w, b = rnd(R, R, 128), rnd(2, R * 32, s), rnd(128, 1024) * 0.05, rnd(128)
    nrm, tail = torch.rand(R, R, generator=g).to(dev) * s, torch.randint(-128, 128, (R, R, 128), generator=g).to(dev, torch.int8)

    def run(r, xt):
        zz, t = z[:r, :r].contiguous(), tail[:r, :r].clone(memory_format=torch.contiguous_format) if xt else None
        out = torch.empty_like(zz)
        _lib.opm_fused(out, zz, ab[0], ab[1], w, b, nrm[:r, :r].contiguous(), r=r, spad=s, eps=1e-3, xtail=t)
        return out, t
    for xt in (False, True):
        whole = run(R, xt)
        a, bb = (ab[i].float().view(R, 32, s) for i in range(2))
        o = torch.einsum("ids,jes->ijed", a[:40].cpu(), bb[:40].cpu()).reshape(40, 40, 1024).to(torch.bfloat16).float()
        ref = z[:40, :40].float().cpu() + (o @ w.float().cpu().t() + b.float().cpu()) / (nrm[:40, :40, None].cpu() + 1e-3)
        assert float((whole[0][:40, :40].float().cpu() - ref).norm() / ref.norm()) < 6e-3
        for r in (32, 128, 160):
            y, t = run(r, xt)
            assert torch.equal(y, whole[0][:r, :r]) and (not xt or torch.equal(t, whole[1][:r, :r])), (r, xt)


@pytest.mark.parametrize("B,N", [(1, 1), (3, 37), (64, 64), (131, 96)])
def test_fp32_channel_major_rows_masked(dev, B, N):
    """A row mask with strides of its own on a channel-major operand, over 32 and 64 rows per workgroup and outputs of either
    order: masked rows are zero, the others are the products (32-bit sums: 1e-5 of the largest)."""
    from fastfold_amd import _lib
    g = torch.Generator().manual_seed(B * N)
    K, M, kp = 128, B * N, (N + 3) // 4 * 4
    xt, w, b = torch.randn(K, B, kp, generator=g), torch.randn(128, K, generator=g) / K ** 0.5, torch.randn(128, generator=g)
    ln, mask = (1 + 0.1 * torch.randn(K, generator=g), 0.1 * torch.randn(K, generator=g)), (torch.rand(N, B, generator=g) > 0.3).float()
    x = xt[:, :, :N].reshape(K, M).t().numpy()
    xt, w, b, mask, ln = xt.to(dev), w.to(dev), b.to(dev), mask.to(dev), tuple(t.to(dev) for t in ln)
    for norm in (True, False):
        out, cm = torch.full((M, 128), 7.0, device=dev), torch.full((128, B * kp), 7.0, device=dev)
        mk = dict(rowmask=mask, m_so=1, m_si=B)
        tiles = [_lib.make_tile(out, bias=b, inner=N, s_o=N * 128, s_i=128, **mk)]
        if norm:
            tiles.append(_lib.make_tile(cm, bias=b, inner=N, s_o=kp, s_i=1, s_h=32 * B * kp, s_d=B * kp, **mk))
        _lib.fused_linear(xt, torch.cat([w, w]), tiles, M=M, K=K, a_inner=N, a_so=kp, a_si=1, a_chanmajor=True, a_cs=B * kp, ln=ln if norm else None)
        ref = ops_np.linear(ops_np.layer_norm(x, *(t.cpu() for t in ln)) if norm else x, w.cpu(), b.cpu()) * _np(mask).T.reshape(M, 1)
        assert np.abs(_np(out) - ref).max() <= 1e-5 * max(np.abs(ref).max(), 1.0)
        if norm:
            assert np.abs(_np(cm).reshape(128, B, kp)[:, :, :N].reshape(128, M).T - ref).max() <= 1e-5 * max(np.abs(ref).max(), 1.0)


@pytest.mark.parametrize("M,nt,ncols", [(33, 1, 64), (9000, 1, 36), (33000, 1, 64), (130000, 1, 20), (131041, 4, 64), (131041, 4, 44)])
def test_fp32_glu_tile_with_residual(dev, M, nt, ncols):
    """GLU channels stored [row][channel] onto a residual, in place, from 32 rows per workgroup to the persistent layout (four tiles):
    the second unit of 32 channels takes the second half of the residual's (against float64; 2e-5 of the largest)."""
    from fastfold_amd import _lib
    g = torch.Generator().manual_seed(M + ncols)
    K = 128
    x, b = torch.randn(M, K, generator=g).to(dev), torch.randn(nt * 128, generator=g).to(dev)
    w, out = (torch.randn(nt * 128, K, generator=g) / K ** 0.5).to(dev), torch.randn(M, nt * 64, generator=g).to(dev)
    ref = out.double().view(M, nt, 64)
    y = (x.double() @ w.double().t() + b).view(M, nt, 2, 2, 32)             # a tile: [p 0..31 | g 0..31 | p 32..63 | g 32..63]
    ref[..., :ncols] += (y[..., 0, :] * torch.sigmoid(y[..., 1, :])).reshape(M, nt, 64)[..., :ncols]
    tiles = [_lib.make_tile(out.data_ptr() + 256 * i, bias=b.data_ptr() + 512 * i, glu=1, ncols=ncols, resid=out.data_ptr() + 256 * i,
                            inner=M, s_i=nt * 64) for i in range(nt)]
    _lib.fused_linear(x, w, tiles, M=M, K=K)
    assert float((out.view(M, nt, 64) - ref).abs().max()) <= 2e-5 * float(ref.abs().max())


@pytest.mark.parametrize("r", [362, 411])
def test_fp32_gated_projection_persistent_layout(dev, r):
    """The GLU projection of a triangle multiplication (channel-major outputs, row mask) at rows enough for the persistent layout
    (131 044: eight units on 256 workgroups of eight waves) and a ragged last slab, against the staged kernel."""
    from fastfold_amd import _lib
    M, K, nt = r * r, 128, 4
    g = torch.Generator(device=dev).manual_seed(r)
    x, w, b = (torch.randn(*sh, device=dev, generator=g) for sh in ((M, K), (nt * 128, K), (nt * 128,)))
    w, ln, mask = w / K ** 0.5, torch.randn(2, K, device=dev, generator=g), (torch.rand(r, device=dev, generator=g) > 0.3).float()
    got = []
    for staged in (True, False):
        got.append(torch.full((256, M), 7.0, device=dev))
        tiles = [_lib.make_tile(got[-1].data_ptr() + 256 * i * M, inner=r, s_o=r, s_i=1, s_h=32 * M, s_d=M, glu=1, ncols=64, bias=b.data_ptr() + 512 * i,
                                rowmask=mask, m_so=1) for i in range(nt)]
        _lib.fused_linear(x, w, tiles, M=M, K=K, ln=(ln[0], ln[1]), staged=staged)
    assert float((got[0] - got[1]).abs().max()) <= 1e-5 * float(got[0].abs().max())


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("K", [64, 128, 256])
def test_value_tile_with_row_mask(dev, dtype, K):
    """A row mask on the v tiles of an attention: masked keys have zeros."""
    from fastfold_amd import _lib
    from fastfold_amd.model.fastnn.kernel import layouts
    B2, N = 5, 96
    g = torch.Generator().manual_seed(K)
    x, w = torch.randn(B2, N, K, generator=g).to(dev, dtype), (torch.randn(128, K, generator=g) / K ** 0.5).to(dev, dtype)
    mask, v = (torch.rand(B2, N, generator=g) > 0.3).to(dev, dtype), torch.zeros(B2, 4, 3, 2, 32, 4, 4, dtype=dtype, device=dev)
    _lib.fused_linear(x, w, [_lib.make_tile(v, kind=_lib.FFK_TILE_V, inner=N, s_o=4 * 3072, s_h=3072, rowmask=mask, m_so=N, m_si=1)], M=B2 * N, K=K)
    ref = (ops_np.linear(_np(x), _np(w)) * _np(mask)[..., None]).reshape(B2, N, 4, 32).transpose(0, 2, 1, 3)
    assert _rel(_np(layouts.untile_v(v, N)), ref) < TOL[dtype]


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("K,chan", [(128, False), (256, False), (128, True)])
@pytest.mark.parametrize("M", [40, 96 * 131 - 24])
def test_value_tile_of_a_launch_that_ends_inside_it(dev, dtype, K, chan, M):
    """Rows of a key tile behind the last row of the launch keep what they hold."""
    from fastfold_amd import _lib
    from fastfold_amd.model.fastnn.kernel import layouts
    N = 96
    B = (M + N - 1) // N
    g = torch.Generator().manual_seed(K + M)
    x, w = torch.randn(B * N, K, generator=g).to(dev, dtype), (torch.randn(128, K, generator=g) / K ** 0.5).to(dev, dtype)
    v = torch.full((B, 4, 3, 2, 32, 4, 4), 7.0, dtype=dtype, device=dev)
    kw = dict(a_chanmajor=True, a_inner=B * N, a_si=1, a_cs=B * N) if chan else {}
    _lib.fused_linear(x.t().contiguous() if chan else x, w, [_lib.make_tile(v, kind=_lib.FFK_TILE_V, inner=N, s_o=4 * 3072, s_h=3072)], M=M, K=K, **kw)
    got = _np(layouts.untile_v(v, N)).transpose(0, 2, 1, 3).reshape(B * N, 128)
    ref = ops_np.linear(_np(x), _np(w))
    assert _rel(got[:M], ref[:M]) < TOL[dtype] and (got[M:] == 7.0).all()
