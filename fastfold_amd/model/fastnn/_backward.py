"""Backward pass of an Evoformer block as launch sequences (the gradients of fastfold/model/fastnn/evoformer.py:64-76).

The block is its own checkpoint: the forward pass keeps m and z only.  ``block_backward`` runs the sub-modules forward once more
with the fused launches, keeping the residual streams between them, and then walks them backwards; each ``*_backward`` function
recomputes what it needs of its sub-module from that sub-module's input and writes

    dx = dy + (gradient of the update for the cotangent dy)

and the gradients of its parameters.  Differentiated operator by operator through autograd, a block at N_seq = 128, N_res = 256
took about 350 launches and 9 ms of them, half of that copies, conversions, strided reductions and elementwise passes between the
products, and as much host time; the sequences below are about 150 launches, recorded and replayed like the forward ones.

Rows are the logical rows of the sub-module (b, n) -> b * N + n; ``a_map = (inner, s_o, s_i)`` addresses them in the tensors of
the natural order, so that the transposed attentions need no transposed copies.  Extents are multiples of 32 (the caller pads).
"""
import functools
import math

import torch

from fastfold_amd import _lib, _plan
from fastfold_amd._lib import FFK_ACT_GATE_POS, FFK_ACT_RELU, FFK_TILE_ACC, FFK_TILE_BIAS, FFK_TILE_V, LOG2E, make_tile
from . import _fused as F_
from ._fused import alloc, es_of, pack_rows, pack_vec, round_up


# ------------------------------------------------------------------------------------------------ pieces ----
def _plain(rows, width):
    """Row map of a [rows, width] matrix."""
    return rows, 0, width


def _rows(x, w, out, *, M, K, N, a_map=None, ln=None, bias=None, act=0, gate=None, gate_ld=0, w_row=0, out_ld=None):
    """out[M, N] (row pitch ``out_ld``) = act(LN(x) W^T + b) over the rows ``a_map`` of x."""
    es = es_of(x.dtype)
    ld = N if out_ld is None else out_ld
    inner, so, si = _plain(M, K) if a_map is None else a_map
    nt = (N + 127) // 128
    per = _lib.WS_TILES
    for t0 in range(0, nt, per):
        tiles = [make_tile(out.data_ptr() + t * 128 * es, bias=None if bias is None else bias.data_ptr() + t * 128 * es,
                           act=act, gate=None if gate is None else gate.data_ptr() + t * 128 * es, gate_ld=gate_ld,
                           inner=M, s_i=ld, ncols=min(128, N - t * 128)) for t in range(t0, min(nt, t0 + per))]
        _lib.fused_linear(x, w, tiles, M=M, K=K, a_inner=inner, a_so=so, a_si=si, ln=ln, w_row_off=w_row + t0 * 128)


def _slices(M, N, K, dtype):
    """Slices of the rows of a weight gradient: two workgroups per CU over its 128 x 128 output tiles, at most 64 MB of partial sums,
    whole 64-row steps and two of them at least.  Small outputs take half the slices: the sums over them cost more than the second
    workgroup saves (us with 512 and 256 workgroups, bf16: 65 536 x 128 x 128 22.3, 18.3, 65 536 x 512 x 128 30.6, 29.1, but
    65 536 x 640 x 128 33.1, 38.9; fp32: 38.2, 35.2, but 93.3, 101.1)."""
    tiles = ((N + 127) // 128) * ((K + 127) // 128)
    steps = (M + 63) // 64
    groups = 256 if tiles <= (4 if dtype == torch.bfloat16 else 1) else 512
    s = max(1, min(groups // tiles, (64 << 20) // (4 * N * K), (steps + 1) // 2))
    return (steps + (steps + s - 1) // s - 1) // ((steps + s - 1) // s)


def _wgrad(out, colsum, y, x, *, M, N, K, dtype, device, y_map=None, x_map=None, **kw):
    s = _slices(M, N, K, dtype)
    ws = alloc((s * N * (K + 1),), torch.float32, device)
    _lib.weight_grad(out, colsum, ws, y, x, M=M, N=N, K=K, slices=s, dtype=dtype, y_map=_plain(M, N) if y_map is None else y_map,
                     x_map=_plain(M, K) if x_map is None else x_map, **kw)


def _ln_back(dx, xn, g, ln_mod, ln, dy, x, resid, *, rows, C):
    ws = alloc((_lib.FFK_LN_BWD_BLOCKS * 2 * C,), torch.float32, x.device)
    _lib.layernorm_bwd_rows(dx, xn, g[ln_mod.weight], g[ln_mod.bias], ws, dy, x, ln[0], ln[1], resid, rows=rows, C=C, dtype=x.dtype)


def distinct(params):
    """Whether no parameter serves in two places: ``Grads`` has one piece for each place, and neither the sum of two nor, for a
    place whose neighbours lie elsewhere, the memory one product writes."""
    return len({id(p) for p in params}) == len(params)


class Grads:
    """Gradients of a module's parameters as pieces of one flat tensor, in the order ``params`` lists them: neighbours in the
    list are neighbours in memory, so one product can write several (the projections of a concatenated operand)."""

    def __init__(self, params):
        self.params = params
        self.offsets, n = {}, 0
        for p in params:
            self.offsets[id(p)] = n
            n += p.numel()
        self.numel = n
        self.flat = None

    def bind(self, flat):
        other = Grads.__new__(Grads)
        other.params, other.offsets, other.numel, other.flat = self.params, self.offsets, self.numel, flat
        return other

    def __getitem__(self, p):
        return self.flat.data_ptr() + self.offsets[id(p)] * self.flat.element_size()

    def views(self):
        return [self.flat[self.offsets[id(p)]:self.offsets[id(p)] + p.numel()].view(p.shape) for p in self.params]


def _att_params(att):
    return [att.to_qkv.weight, att.gating_linear.weight]


def row_parameters(row):
    return [row.layernormM.weight, row.layernormM.bias, row.layernormZ.weight, row.layernormZ.bias, row.linear_b_weights,
            *_att_params(row.attention), row.attention.gating_bias, row.attention.o_linear.weight, row.out_bias]


def column_parameters(col):
    return [col.layernormM.weight, col.layernormM.bias, *_att_params(col.attention), col.attention.gating_bias,
            col.attention.o_linear.weight, col.attention.o_linear.bias]


def transition_parameters(tr):
    return [tr.norm.weight, tr.norm.bias, tr.linear1.weight, tr.linear1.bias, tr.linear2.weight, tr.linear2.bias]


def outer_product_mean_parameters(opm):
    return [opm.layernormM.weight, opm.layernormM.bias, opm.linear_a.weight, opm.linear_b.weight, opm.linear_a.bias,
            opm.linear_b.bias, opm.o_linear.weight, opm.o_linear.bias]


def triangle_multiplication_parameters(tm):
    return [tm.layernorm1.weight, tm.layernorm1.bias, tm.left_right_projection.weight, tm.left_right_gate.weight,
            tm.output_gate.weight, tm.left_right_projection.bias, tm.left_right_gate.bias, tm.output_gate.bias,
            tm.layernorm2.weight, tm.layernorm2.bias, tm.output_projection.weight, tm.output_bias]


def triangle_attention_parameters(ta):
    return [ta.layernorm1.weight, ta.layernorm1.bias, *_att_params(ta.attention), ta.linear_b.weight,
            ta.attention.gating_bias, ta.attention.o_linear.weight, ta.out_bias]


def parameters(block):
    """Every parameter of the block (``as_built``), grouped for ``Grads``."""
    msa, pair = block.msa, block.pair
    return [*row_parameters(msa.MSARowAttentionWithPairBias), *column_parameters(msa.MSAColumnAttention),
            *transition_parameters(msa.MSATransition), *transition_parameters(pair.PairTransition),
            *outer_product_mean_parameters(block.communication),
            *triangle_multiplication_parameters(pair.TriangleMultiplicationOutgoing),
            *triangle_multiplication_parameters(pair.TriangleMultiplicationIncoming),
            *triangle_attention_parameters(pair.TriangleAttentionStartingNode),
            *triangle_attention_parameters(pair.TriangleAttentionEndingNode)]


# Which modules the sequences below cover: by widths (the Evoformer's own; the narrower heads and rows of the feeder stacks are
# differentiated operator by operator through autograd), by the dtype of their input, and only with sub-modules as they were
# constructed.  The sequences read the parameters of the sub-modules and never call them, so that a hook, a replaced forward or
# an adapter in the place of a Linear would not be seen.
def _dtype_ok(*ts):
    return ts[0].dtype in (torch.bfloat16, torch.float32) and all(t.dtype == ts[0].dtype and t.is_cuda for t in ts)


@functools.lru_cache(maxsize=None)
def _anatomy():
    """The classes the sequences stand for, with the names of their sub-modules and parameters."""
    from . import msa, ops, triangle
    wb, norm_linears = {"weight", "bias"}, {"norm", "linear1", "linear2"}
    tm = {"layernorm1", "layernorm2", "left_right_projection", "left_right_gate", "output_gate", "output_projection"}, {"output_bias"}
    ta = {"layernorm1", "linear_b", "attention"}, {"out_bias"}
    return {ops.Linear: (set(), wb), ops.LayerNorm: (set(), wb),
            ops.SelfAttention: ({"to_qkv", "gating_linear", "o_linear"}, {"gating_bias"}),
            ops.Transition: (norm_linears, set()), ops.ChunkTransition: (norm_linears, set()),
            ops.OutProductMean: ({"layernormM", "linear_a", "linear_b", "o_linear"}, set()),
            ops.AsyncChunkTriangleMultiplicationOutgoing: tm, ops.AsyncChunkTriangleMultiplicationIncoming: tm,
            ops.ChunkTriangleAttentionStartingNode: ta, ops.ChunkTriangleAttentionEndingNode: ta,
            msa.MSARowAttentionWithPairBias: ({"layernormM", "layernormZ", "attention"}, {"linear_b_weights", "out_bias"}),
            msa.MSAColumnAttention: ({"layernormM", "attention"}, set()),
            msa.MSACore: ({"MSARowAttentionWithPairBias", "MSAColumnAttention", "MSATransition"}, set()),
            triangle.PairCore: ({"TriangleMultiplicationOutgoing", "TriangleMultiplicationIncoming", "TriangleAttentionStartingNode",
                                 "TriangleAttentionEndingNode", "PairTransition"}, set())}


def _as_built(mod, anatomy):
    d = mod.__dict__
    parts, params = anatomy.get(type(mod), (None, None))
    return (d["_modules"].keys() == parts and d["_parameters"].keys() == params and "forward" not in d
            and not (d["_forward_hooks"] or d["_forward_pre_hooks"] or d["_backward_hooks"] or d["_backward_pre_hooks"])
            and d.get("eps", 1e-5) == 1e-5 and all([_as_built(c, anatomy) for c in d["_modules"].values()]))


def as_built(mod):
    """Whether everything below ``mod`` is as it was constructed and without hooks."""
    anatomy = _anatomy()
    return not torch.nn.modules.module._has_any_global_hook() and all([_as_built(c, anatomy) for c in mod._modules.values()])


def _covers_attention(att, d):
    return att.gating and att.c == 32 and att.n_head * 32 == d and att.out_dim == d and att.qkv_dim == d and d in (128, 256)


def covers_row(row):
    return _covers_attention(row.attention, row.d_node) and row.d_pair == 128 and row.n_head <= 8


def covers_column(col):
    return _covers_attention(col.attention, col.d_node) and col.attention.o_linear.use_bias


def covers_transition(tr):
    return tr.linear1.in_features in (128, 256) and tr.linear1.out_features % 128 == 0


def covers_outer_product_mean(opm):
    return opm.n_feat_proj == 32 and opm.o_linear.out_features == 128 and opm.linear_a.in_features in (64, 128, 256)


def covers_triangle_multiplication(tm):
    return tm.c == 128 and tm.d_pair == 128


def covers_triangle_attention(ta):
    return _covers_attention(ta.attention, ta.d_pair) and ta.n_head <= 4


def supported(block, params):
    """Whether ``block_backward`` covers this block (if it is ``as_built``); ``params``: its ``parameters``."""
    msa, pair = block.msa, block.pair
    return (covers_row(msa.MSARowAttentionWithPairBias) and covers_column(msa.MSAColumnAttention)
            and covers_transition(msa.MSATransition) and covers_transition(pair.PairTransition)
            and covers_outer_product_mean(block.communication)
            and covers_triangle_multiplication(pair.TriangleMultiplicationOutgoing)
            and covers_triangle_multiplication(pair.TriangleMultiplicationIncoming)
            and covers_triangle_attention(pair.TriangleAttentionStartingNode)
            and covers_triangle_attention(pair.TriangleAttentionEndingNode)
            and distinct(params))


# -------------------------------------------------------------------------------------------- transition ----
def transition_backward(tr, x, dy, dx, g):
    M, C = x.shape
    H = tr.linear1.out_features
    dt, dev = x.dtype, x.device
    ln = _ln(tr.norm, dt)
    w1, b1, w2t, w1t = tr._packed(("tr_bwd", dt, dev), [tr.linear1.weight, tr.linear1.bias, tr.linear2.weight], lambda: (
        pack_rows([tr.linear1.weight], dt, dev), pack_vec([tr.linear1.bias], dt, dev), pack_rows([tr.linear2.weight.t()], dt, dev),
        tr.linear1.weight.detach().to(dt).t().contiguous()))
    h = alloc((M, H), dt, dev)
    _rows(x, w1, h, M=M, K=C, N=H, ln=ln, bias=b1, act=FFK_ACT_RELU)
    dh = alloc((M, H), dt, dev)
    _rows(dy, w2t, dh, M=M, K=C, N=H, act=FFK_ACT_GATE_POS, gate=h, gate_ld=H)
    dn, xn = alloc((M, C), dt, dev), alloc((M, C), dt, dev)
    _lib.bgemm_nt(dh, w1t, dn, M=M, N=C, K=H, lda=H, ldb=H)
    _wgrad(g[tr.linear2.weight], g[tr.linear2.bias], dy, h, M=M, N=C, K=H, dtype=dt, device=dev)
    _ln_back(dx, xn, g, tr.norm, ln, dn, x, dy, rows=M, C=C)
    _wgrad(g[tr.linear1.weight], g[tr.linear1.bias], dh, xn, M=M, N=H, K=C, dtype=dt, device=dev)


def _ln(ln, dt):
    return ln.weight.detach().to(dt).contiguous(), ln.bias.detach().to(dt).contiguous()


# --------------------------------------------------------------------------------------------- attention ----
def attention_backward(owner, att, ln_mod, x, dy, dx, g, out_bias, *, B2, N, a_map, kb, flags, bias_t=None, bias_padded=False,
                       linear_b=None, drop=None, drop_map=None):
    """Gated attention over N tokens for each of B2 rows, residual from its own input x.  The additive bias is either given
    (``bias_t``, tiles) or produced from the same rows by ``linear_b``.  Returns the partial sums of its gradient and their
    number, ([parts, H, N, N] fp32), for a given bias; the gradient of ``linear_b`` is part of this function."""
    C, H = att.qkv_dim, att.n_head
    HC, M, dt, dev = H * 32, B2 * N, x.dtype, x.device
    es, NT = es_of(dt), N // 32
    inner, so, si = a_map
    ln = _ln(ln_mod, dt)
    Kd = 4 * HC + (32 if linear_b is not None else 0)

    def build():
        q, k, v = att.to_qkv.weight.detach().unflatten(0, (3, HC))
        gw = att.gating_linear.weight.detach()
        extra = [] if linear_b is None else [torch.nn.functional.pad(linear_b.weight.detach(), (0, 0, 0, 32 - linear_b.out_features))]
        return (pack_rows([q, q, k, k] + extra, dt, dev), pack_rows([v, v, gw], dt, dev),
                pack_vec([att.gating_bias], dt, dev), pack_rows([att.o_linear.weight.t()], dt, dev),
                torch.cat([q, k, v, gw] + extra, 0).to(dt).t().contiguous())
    ps = [att.to_qkv.weight, att.gating_linear.weight, att.gating_bias, att.o_linear.weight]
    w_qk, w_vg, gb, wo_t, wcat_t = owner._packed(("att_bwd", dt, dev), ps + ([] if linear_b is None else [linear_b.weight]), build)

    # operand tiles and the gate's pre-activation, as in the forward pass; q, k and v in both orders
    tiles = {n: alloc((B2, H, NT, 1024), dt, dev) for n in ("q_t", "q_v", "k_t", "k_v", "v_t", "v_v")}
    gpre = alloc((M, HC), dt, dev)
    tkw = dict(inner=N, s_o=H * NT * 1024, s_h=NT * 1024)
    qscale = LOG2E / math.sqrt(32.0)

    def op_tiles(name, kind, scale=1.0):
        return [make_tile(tiles[name].data_ptr() + t * 4 * NT * 1024 * es, kind=kind, scale=scale, **tkw) for t in range(HC // 128)]
    akw = dict(M=M, K=C, a_inner=inner, a_so=so, a_si=si, ln=ln)
    first = [*op_tiles("q_t", FFK_TILE_ACC, qscale), *op_tiles("q_v", FFK_TILE_V, qscale), *op_tiles("k_t", FFK_TILE_ACC),
             *op_tiles("k_v", FFK_TILE_V)]
    if linear_b is not None:
        bias_padded = True
        bias_t = alloc((H, NT, NT + 1, 1024), dt, dev)
        first.append(make_tile(bias_t, kind=FFK_TILE_BIAS, inner=N, s_o=(NT + 1) * 1024, s_h=NT * (NT + 1) * 1024, ncols=H, scale=LOG2E))
    gates = [make_tile(gpre.data_ptr() + t * 128 * es, inner=M, s_i=HC) for t in range(HC // 128)]
    second = [*op_tiles("v_t", FFK_TILE_ACC), *op_tiles("v_v", FFK_TILE_V), *gates]
    per = _lib.WS_TILES if C == 256 else _lib.FFK_MAX_TILES
    for w, ts in ((w_qk, first), (w_vg, second)):
        for t0 in range(0, len(ts), per):
            _lib.fused_linear(x, w, ts[t0:t0 + per], w_row_off=t0 * 128, **akw)
    o, lse = alloc((M, HC), dt, dev), alloc((B2 * H * N,), torch.float32, dev)
    _lib.attention_fwd_lse(o, lse, tiles["q_t"], tiles["k_t"], tiles["v_v"], bias_t, kb, flags, B2=B2, H=H, N=N, bias_padded=bias_padded)

    if drop is not None:
        dyd = alloc((M, C), dt, dev)
        _lib.scale_rows(dyd, dy, drop, rows=M, C=C, inner=drop_map[0], m_so=drop_map[1], m_si=drop_map[2], mode=0, dtype=dt)
    else:
        dyd = dy
    dgo = alloc((M, HC), dt, dev)
    _rows(dyd, wo_t, dgo, M=M, K=C, N=HC, a_map=a_map)
    cat = alloc((M, Kd), dt, dev)                        # [dq | dk | dv | d gate | d bias] rows
    go, do_t, do_v = alloc((M, HC), dt, dev), alloc((B2, H, NT, 1024), dt, dev), alloc((B2, H, NT, 1024), dt, dev)
    dsum = alloc((B2 * H * N,), torch.float32, dev)
    at = cat.data_ptr()
    _lib.att_gate_bwd(go, at + 3 * HC * es, do_t, do_v, dsum, dgo, gpre, gb, o, B2=B2, N=N, H=H, g_ld=HC, dg_ld=Kd, dtype=dt)
    parts = max(1, min((4096 + H * NT * NT - 1) // (H * NT * NT), (B2 + 7) // 8)) if bias_t is not None else 0
    dbias = alloc((parts, H, N, N), torch.float32, dev) if parts else None
    _lib.attention_bwd_rows(at, at + HC * es, at + 2 * HC * es, dbias, lse, dsum, tiles["q_t"], tiles["q_v"], tiles["k_t"],
                            tiles["k_v"], tiles["v_t"], bias_t, kb, do_t, do_v, B2=B2, H=H, N=N, s_b=N * Kd, s_h=32, s_n=Kd,
                            dq_scale=1.0 / math.sqrt(32.0), dk_scale=1.0 / LOG2E, dtype=dt, dbias_parts=parts, bias_padded=bias_padded)
    if linear_b is not None:
        _lib.bias_cols(at + 4 * HC * es, dbias, parts=parts, rows=M, H=H, ld=Kd, dtype=dt)
    dn, xn = alloc((M, C), dt, dev), alloc((M, C), dt, dev)
    _lib.bgemm_nt(cat, wcat_t, dn, M=M, N=C, K=Kd, lda=Kd, ldb=Kd, inner=inner, s_o=so, s_i=si)
    _wgrad(g[att.o_linear.weight], g[out_bias], dyd, go, M=M, N=C, K=HC, dtype=dt, device=dev, y_map=a_map)
    _ln_back(dx, xn, g, ln_mod, ln, dn, x, dy, rows=M, C=C)
    _wgrad(g[att.to_qkv.weight], g[att.gating_bias], cat, xn, M=M, N=Kd, K=C, dtype=dt, device=dev, x_map=a_map,
           n_out=4 * HC + (0 if linear_b is None else linear_b.out_features), cs_first=3 * HC, cs_count=HC)
    return dbias, parts


def row_attention_backward(row, m, z, dy, dm, dz_in, dz, g, *, s, r, kb, flags, drop):
    """MSA row attention with pair bias: dm for the cotangent dy, and dz = dz_in + what the bias passes on."""
    dt, dev = m.dtype, m.device
    Cz, H = row.d_pair, row.n_head
    lnz = _ln(row.layernormZ, dt)
    wb, wb_t = row._packed(("wb_bwd", dt, dev), [row.linear_b_weights], lambda: (
        pack_rows([row.linear_b_weights], dt, dev),
        torch.nn.functional.pad(row.linear_b_weights.detach(), (0, 0, 0, 32 - H)).to(dt).t().contiguous()))
    pbs = row._packed(("pbs", dt, dev), [row.linear_b_weights, row.layernormZ.weight, row.layernormZ.bias],
                      lambda: F_.PairBiasScratch(Cz, dev))
    bias_t = F_.pair_bias(z, r=r, C=Cz, H=H, ln=lnz, wb_pk=wb, pb_scratch=pbs)
    dbias, parts = attention_backward(row, row.attention, row.layernormM, m, dy, dm, g, row.out_bias, B2=s, N=r,
                                      a_map=_plain(s * r, row.d_node), kb=kb, flags=flags, bias_t=bias_t,
                                      drop=drop, drop_map=(r, 0, row.d_node))
    P = r * r
    db = alloc((P, 32), dt, dev)
    _lib.bias_cols(db, dbias, parts=parts, rows=P, H=H, ld=32, dtype=dt)
    dn, zn = alloc((P, Cz), dt, dev), alloc((P, Cz), dt, dev)
    _lib.bgemm_nt(db, wb_t, dn, M=P, N=Cz, K=32, lda=32, ldb=32)
    _ln_back(dz, zn, g, row.layernormZ, lnz, dn, z, dz_in, rows=P, C=Cz)
    _wgrad(g[row.linear_b_weights], None, db, zn, M=P, N=32, K=Cz, dtype=dt, device=dev, n_out=H)


# ------------------------------------------------------------------------------- triangle multiplication ----
def triangle_multiplication_backward(tm, z, dy, dx, g, *, r, mask, drop):
    C = c = 128
    M, dt, dev = r * r, z.dtype, z.device
    es = es_of(dt)
    incoming = tm._incoming
    ln1, ln2 = _ln(tm.layernorm1, dt), _ln(tm.layernorm2, dt)
    ps = [tm.left_right_projection.weight, tm.left_right_projection.bias, tm.left_right_gate.weight, tm.left_right_gate.bias,
          tm.output_gate.weight, tm.output_gate.bias, tm.output_projection.weight, tm.output_bias]

    def build():
        w, b, n_glu = F_.pack_trimul(*ps[:6], c, dt, dev)
        return (w, b, n_glu, pack_rows([ps[2], ps[4]], dt, dev), pack_vec([ps[3], ps[5]], dt, dev), pack_rows([ps[6]], dt, dev),
                pack_vec([ps[7]], dt, dev), pack_rows([ps[6].t()], dt, dev),
                torch.cat([ps[0].detach(), ps[2].detach(), ps[4].detach()], 0).to(dt).t().contiguous())
    w_glu, b_glu, n_glu, w_g, b_g, w_out, b_out, w_out_t, wcat_t = tm._packed(("tm_bwd", dt, dev), ps, build)
    # the gated projections channel-major as in the forward pass, and the gates' pre-activations as rows
    kpad = r
    cs = r * kpad + F_._TRIMUL_CHAN_PAD
    lr = alloc((2, c, cs), dt, dev)
    a_map, m_so, m_si = ((r, C, r * C), 1, r) if incoming else ((M, 0, C), r, 1)
    tiles = []
    for side in range(2):
        for t in range(c // 64):
            ti = side * (c // 64) + t
            tiles.append(make_tile(lr.data_ptr() + (side * c + t * 64) * cs * es, bias=b_glu.data_ptr() + ti * 128 * es, glu=1, ncols=64,
                                   inner=r, s_o=kpad, s_i=1, s_h=32 * cs, s_d=cs, rowmask=mask, m_so=m_so, m_si=m_si))
    _lib.fused_linear(z, w_glu, tiles, M=M, K=C, a_inner=a_map[0], a_so=a_map[1], a_si=a_map[2], ln=ln1)
    pg = alloc((M, 384), dt, dev)                        # [gate left | gate right | output gate]
    _rows(z, w_g, pg, M=M, K=C, N=384, ln=ln1, bias=b_g)
    p = alloc((c, cs), dt, dev)
    _lib.bgemm_nt(lr[0], lr[1], p, M=r, N=r, K=kpad, lda=kpad, ldb=kpad, batch=c, a_bs=cs, b_bs=cs, o_bs=cs, s_i=kpad)
    pt = alloc((M, c), dt, dev)
    _lib.transpose_batched(pt, p, B=r, X=c, Y=r, in_bs=kpad, in_xs=cs, out_bs=r * c, out_ys=c)
    ab = alloc((M, C), dt, dev)
    _rows(pt, w_out, ab, M=M, K=c, N=C, ln=ln2, bias=b_out)

    dpg = alloc((M, 640), dt, dev)                       # [d proj | d gate | d output gate] rows
    dab = alloc((M, C), dt, dev)
    _lib.trimul_gate_bwd(dab, dpg.data_ptr() + 512 * es, dy, drop, ab, pg.data_ptr() + 256 * es, rows=M, C=C, period=r, g_ld=384,
                         dg_ld=640, dtype=dt)
    dn, pn, dpt = alloc((M, c), dt, dev), alloc((M, c), dt, dev), alloc((M, c), dt, dev)
    _rows(dab, w_out_t, dn, M=M, K=C, N=c)
    _ln_back(dpt, pn, g, tm.layernorm2, ln2, dn, pt, None, rows=M, C=c)
    _wgrad(g[tm.output_projection.weight], g[tm.output_bias], dab, pn, M=M, N=C, K=c, dtype=dt, device=dev)
    # dL[i, k] = sum_j dp[i, j] R[j, k],  dR[j, k] = sum_i dp[i, j] L[i, k]: one batch of 2 c products over [dp^T; dp] and
    # [L^T; R^T]
    d2, t2, dlr = alloc((2, c, cs), dt, dev), alloc((2, c, cs), dt, dev), alloc((2, c, cs), dt, dev)
    _lib.transpose_batched(d2[0], dpt, B=r, X=r, Y=c, in_bs=c, in_xs=r * c, out_bs=kpad, out_ys=cs)
    _lib.transpose_batched(d2[1], dpt, B=r, X=r, Y=c, in_bs=r * c, in_xs=c, out_bs=kpad, out_ys=cs)
    _lib.transpose_batched(t2, lr, B=2 * c, X=r, Y=r, in_bs=cs, in_xs=kpad, out_bs=cs, out_ys=kpad)
    _lib.bgemm_nt(d2, t2, dlr, M=r, N=r, K=kpad, lda=kpad, ldb=kpad, batch=2 * c, a_bs=cs, b_bs=cs, o_bs=cs, s_i=kpad)
    for side, d in ((0, dlr[1]), (1, dlr[0])):
        _lib.glu_bwd(dpg.data_ptr() + side * 128 * es, dpg.data_ptr() + (256 + side * 128) * es, d, lr[side],
                     pg.data_ptr() + side * 128 * es, mask, R=r, C=c, cs=cs, kpad=kpad, d_ld=640, g_ld=384,
                     r_i=1 if incoming else r, r_k=r if incoming else 1, dtype=dt)
    dzn, zn = alloc((M, C), dt, dev), alloc((M, C), dt, dev)
    _lib.bgemm_nt(dpg, wcat_t, dzn, M=M, N=C, K=640, lda=640, ldb=640)
    _ln_back(dx, zn, g, tm.layernorm1, ln1, dzn, z, dy, rows=M, C=C)
    _wgrad(g[tm.left_right_projection.weight], g[tm.left_right_projection.bias], dpg, zn, M=M, N=640, K=C, dtype=dt, device=dev)


# ------------------------------------------------------------------------------------ outer product mean ----
def outer_product_mean_backward(opm, m, mask, dz, dm_in, dm, g, *, s, r, nrm, budget, eps=1e-3):
    """dm = dm_in + the gradient of the MSA tensor for the pair cotangent dz (which itself passes on unchanged)."""
    C, Cz, P = m.shape[-1], dz.shape[-1], r * r
    dt, dev = m.dtype, m.device
    es = es_of(dt)
    ln = _ln(opm.layernormM, dt)

    def build():
        wab = torch.cat([opm.linear_a.weight.detach(), opm.linear_b.weight.detach()], 0)
        return (pack_rows([wab], dt, dev), pack_vec([opm.linear_a.bias, opm.linear_b.bias], dt, dev),
                pack_rows([opm.o_linear.weight.t()], dt, dev), wab.to(dt).t().contiguous())
    wab, bab, wo_t, wab_t = opm._packed(("opm_bwd", dt, dev), [opm.linear_a.weight, opm.linear_a.bias, opm.linear_b.weight,
                                                               opm.linear_b.bias, opm.o_linear.weight], build)
    R = r * 32
    ab = alloc((2, R, s), dt, dev)                       # row = residue * 32 + channel
    tile = make_tile(ab, bias=bab, ncols=64, inner=s, s_o=32 * s, s_i=1, s_h=R * s, s_d=s, rowmask=mask, m_so=1, m_si=r)
    _lib.fused_linear(m, wab, [tile], M=s * r, K=C, a_inner=s, a_so=C, a_si=r * C, ln=ln)
    bt = alloc((s, R), dt, dev)
    _lib.transpose_batched(bt, ab[1], B=1, X=R, Y=s, in_bs=0, in_xs=s, out_bs=0, out_ys=R)
    du = alloc((P, Cz), dt, dev)
    _lib.scale_rows(du, dz, nrm, rows=P, C=Cz, inner=P, m_so=0, m_si=1, mode=2, eps=eps, dtype=dt)
    dab = alloc((r * s, 64), dt, dev)                    # row (i, s'): d of the projections a | b of that residue and sequence
    ci = max(1, min(r, budget // (r * 2048 * es)))       # residues i per piece: two [ci * r, 1024] intermediates
    O, dO = alloc((ci * r, 1024), dt, dev), alloc((ci * 32, R), dt, dev)
    # d Wo and d b are sums over the pieces; d a is complete in each: a sum over a whole row of dO, cut into four parts because
    # its [32 ci, s] output alone is too few tiles
    acc_o, acc_b = (alloc((n,), torch.float32, dev) for n in (Cz * 1024 + Cz, R * s)) if ci < r else (None, None)
    ks = 4 if R % 128 == 0 else 1
    da = alloc((ks, ci * 32, s), torch.float32, dev)
    for i0 in range(0, r, ci):
        n = min(ci, r - i0)
        a_i = ab.data_ptr() + i0 * 32 * s * es
        du_i = du.data_ptr() + i0 * r * Cz * es
        flags = (_lib.FFK_WGRAD_READ if i0 else 0) | (_lib.FFK_WGRAD_WRITE if i0 + n < r else 0)
        _lib.bgemm_nt(a_i, ab[1], O, M=32 * n, N=R, K=s, lda=s, ldb=s, inner=32, s_o=r * 1024, s_i=32, s_h=1024, s_d=1, dtype=dt)
        _wgrad(g[opm.o_linear.weight], g[opm.o_linear.bias], du_i, O, M=n * r, N=Cz, K=1024, dtype=dt, device=dev, acc=acc_o, flags=flags)
        # d O as the matrix [(i, d)][(j, e)]: column 32 d + e of row (i, j)
        for t0 in range(0, 8, 4):
            tiles = [make_tile(dO.data_ptr() + t * 4 * R * es, inner=r, s_o=32 * R, s_i=32, s_h=R) for t in range(t0, t0 + 4)]
            _lib.fused_linear(du, wo_t, tiles, M=n * r, K=Cz, a_off=i0 * r * Cz, w_row_off=t0 * 128)
        _lib.bgemm_nt(dO, bt, da, M=32 * n, N=s, K=R // ks, lda=R, ldb=R, batch=ks, a_bs=R // ks, b_bs=R // ks, o_bs=32 * n * s, s_i=s,
                      out_f32=True, dtype=dt)
        _lib.slice_sum(dab.data_ptr() + i0 * s * 64 * es, da, slices=ks, N=32 * n, K=s, o_map=(32, s * 64, 1, 64), dtype=dt)
        _wgrad(dab.data_ptr() + 32 * es, None, dO, a_i, M=32 * n, N=R, K=s, dtype=dt, device=dev, o_map=(32, s * 64, 1, 64),
               acc=acc_b, flags=flags)
    _lib.scale_rows(dab, dab, mask, rows=r * s, C=64, inner=s, m_so=1, m_si=r, mode=1, dtype=dt)
    dn, mn = alloc((s * r, C), dt, dev), alloc((s * r, C), dt, dev)
    nat = (s, C, r * C)                                  # row (i, s') of the tensors in m's order
    _lib.bgemm_nt(dab, wab_t, dn, M=r * s, N=C, K=64, lda=64, ldb=64, inner=s, s_o=C, s_i=r * C)
    _ln_back(dm, mn, g, opm.layernormM, ln, dn, m, dm_in, rows=s * r, C=C)
    _wgrad(g[opm.linear_a.weight], g[opm.linear_a.bias], dab, mn, M=r * s, N=64, K=C, dtype=dt, device=dev, x_map=nat)


# ------------------------------------------------------------------------------------ modules on their own ----
def _pad(t, d1, d2):
    """[1, a, b, c] (or a mask [1, a, b]) padded by d1 rows and d2 columns of zeros."""
    if t is None or (d1 == 0 and d2 == 0):
        return t
    return torch.nn.functional.pad(t, (0, 0, 0, d2, 0, d1) if t.dim() == 4 else (0, d2, 0, d1))


def _over(n):
    return round_up(n, 32) - n


def kept(t, like):
    """A mask or dropout multiplier as an autograd function keeps it: in the type of ``like``, contiguous.  Through
    ``save_for_backward``, so that a change of it between the passes is noticed; a tensor made under ``torch.inference_mode``
    cannot be saved and is copied."""
    if t is None:
        return None
    t = t.to(like.dtype).contiguous()
    return t.clone() if t.is_inference() else t


class _Module(torch.autograd.Function):
    """A sub-module under autograd: the fused forward launches, and the backward sequence above at extents padded to whole tiles.
    ``forward(ctx, step, (n_inputs, n_kept), *inputs, *kept, *parameters)``: ``kept`` are the masks and dropout multipliers."""

    @staticmethod
    def forward(ctx, step, counts, *args):
        n, k = counts
        inputs = [t.contiguous() for t in args[:n]]
        ctx.step, ctx.counts, ctx.params = step, counts, args[n + k:]
        ctx.save_for_backward(*inputs, *args[n:])
        return step.forward(*inputs, *args[n:n + k])

    @staticmethod
    def backward(ctx, dy):
        n, k = ctx.counts
        g = Grads(list(ctx.params))
        saved = ctx.saved_tensors[:n + k]                 # raises if one of them, or a parameter, was changed in place
        g = g.bind(torch.empty(g.numel, dtype=dy.dtype, device=dy.device))
        with torch.no_grad():
            dx = ctx.step.backward(dy.contiguous(), g, *saved)
        need = ctx.needs_input_grad[2:]
        return (None, None, *(d if need[i] else None for i, d in enumerate(dx)), *(None for _ in range(k)),
                *(v.to(p.dtype) if need[n + k + i] else None for i, (p, v) in enumerate(zip(ctx.params, g.views()))))


def _apply(step, inputs, extra, params):
    """None: the module's operators have to do it."""
    if not distinct(params):
        return None
    return _Module.apply(step, (len(inputs), len(extra)), *inputs, *(kept(t, inputs[0]) for t in extra), *params)


def _tiles(t):
    """Extents to add to a module's own forward pass: whole tiles in bf16, as in a block (see ``_fused.pad_to_tiles``)."""
    return (_over(t.shape[1]), _over(t.shape[2])) if t.dtype == torch.bfloat16 else (0, 0)


class _TransitionStep:
    def __init__(self, tr):
        self.mod = tr

    def forward(self, x):
        return self.mod._run(x, torch.empty_like(x))

    def backward(self, dy, g, x):
        dx = torch.empty_like(x)
        C = x.shape[-1]
        transition_backward(self.mod, x.view(-1, C), dy.view(-1, C), dx.view(-1, C), g)
        return (dx,)


class _TriMulStep:
    def __init__(self, tm):
        self.mod = tm

    def forward(self, z, mask, drop):
        r = z.shape[1]
        d, _ = _tiles(z)
        z, mask = _pad(z, d, d), _pad(mask, d, d)
        if drop is not None:
            drop = _pad(drop, *((d, 0) if drop.shape[1] == r and drop.shape[2] == 1 else (0, d)))
        return self.mod._run(z, mask, torch.empty_like(z), drop=drop)[:, :r, :r].contiguous()

    def backward(self, dy, g, z, mask, drop):
        r, C = z.shape[1], z.shape[3]
        d = _over(r)
        zp, dyp, mask = _pad(z, d, d), _pad(dy, d, d), _pad(mask, d, d)
        dx = torch.empty_like(zp)
        drop = None if drop is None else _pad(drop, 0, d).reshape(-1, C).contiguous()
        triangle_multiplication_backward(self.mod, zp.view(-1, C), dyp.view(-1, C), dx.view(-1, C), g, r=r + d, mask=mask[0], drop=drop)
        return (dx[:, :r, :r].contiguous(),)


class _TriAttStep(_TriMulStep):
    def backward(self, dy, g, z, mask, drop):
        ta = self.mod
        r, C = z.shape[1], z.shape[3]
        d = _over(r)
        n = r + d
        zp, dyp, mask = _pad(z, d, d), _pad(dy, d, d), _pad(mask, d, d)
        dx = torch.empty_like(zp)
        a_map, sb, sn, dmap = ((n, C, n * C), 1, n, (n, C, 0)) if ta._ending else ((n * n, 0, C), n, 1, (n, 0, C))
        if drop is not None:
            drop = (_pad(drop, d, 0) if ta._ending else _pad(drop, 0, d)).reshape(-1, C).contiguous()
        kb, flags = F_.key_bias(mask[0], z.device, B2=n, N=n, mask_sb=sb, mask_sn=sn)
        attention_backward(ta, ta.attention, ta.layernorm1, zp.view(-1, C), dyp.view(-1, C), dx.view(-1, C), g, ta.out_bias, B2=n, N=n,
                           a_map=a_map, kb=kb, flags=flags, linear_b=ta.linear_b, drop=drop, drop_map=dmap)
        return (dx[:, :r, :r].contiguous(),)


class _ColumnStep:
    def __init__(self, col):
        self.mod = col

    def forward(self, m, mask):
        _, s, r, _ = m.shape
        ds, dr = _tiles(m)
        m, mask = _pad(m, ds, dr), _pad(mask, ds, dr)
        return self.mod._run(m, mask, torch.empty_like(m))[:, :s, :r].contiguous()

    def backward(self, dy, g, m, mask):
        col = self.mod
        _, s, r, C = m.shape
        ds, dr = _over(s), _over(r)
        mp, dyp, mask = _pad(m, ds, dr), _pad(dy, ds, dr), _pad(mask, ds, dr)
        dx = torch.empty_like(mp)
        sp, rp = s + ds, r + dr
        kb, flags = F_.key_bias(mask[0], m.device, B2=rp, N=sp, mask_sb=1, mask_sn=rp)
        attention_backward(col, col.attention, col.layernormM, mp.view(-1, C), dyp.view(-1, C), dx.view(-1, C), g,
                           col.attention.o_linear.bias, B2=rp, N=sp, a_map=(sp, C, rp * C), kb=kb, flags=flags)
        return (dx[:, :s, :r].contiguous(),)


class _RowStep:
    def __init__(self, row):
        self.mod = row

    def forward(self, m, z, mask, drop):
        _, s, r, _ = m.shape
        ds, dr = _tiles(m)
        m, z, mask = _pad(m, ds, dr), _pad(z, dr, dr), _pad(mask, ds, dr)
        return self.mod._run(m, z, mask, torch.empty_like(m), drop=_pad(drop, 0, dr))[:, :s, :r].contiguous()

    def backward(self, dy, g, m, z, mask, drop):
        _, s, r, C = m.shape
        Cz = z.shape[-1]
        ds, dr = _over(s), _over(r)
        mp, dyp, zp, mask = _pad(m, ds, dr), _pad(dy, ds, dr), _pad(z, dr, dr), _pad(mask, ds, dr)
        dm, dz = torch.empty_like(mp), torch.empty_like(zp)
        sp, rp = s + ds, r + dr
        kb, flags = F_.key_bias(mask[0], m.device, B2=sp, N=rp, mask_sb=rp, mask_sn=1)
        drop = None if drop is None else _pad(drop, 0, dr).reshape(-1, C).contiguous()
        row_attention_backward(self.mod, mp.view(-1, C), zp.view(-1, Cz), dyp.view(-1, C), dm.view(-1, C), None, dz.view(-1, Cz), g, s=sp,
                               r=rp, kb=kb, flags=flags, drop=drop)
        return dm[:, :s, :r].contiguous(), dz[:, :r, :r].contiguous()


class _OuterStep:
    def __init__(self, opm, budget):
        self.mod, self.budget = opm, budget

    def forward(self, m, z, mask):
        r = z.shape[1]
        ds, dr = _tiles(m)
        m, z, mask = _pad(m, ds, dr), _pad(z, dr, dr), _pad(mask, ds, dr)
        return self.mod._run(m, mask, z, torch.empty_like(z))[:, :r, :r].contiguous()

    def backward(self, dy, g, m, z, mask):
        _, s, r, C = m.shape
        Cz = z.shape[-1]
        ds, dr = _over(s), _over(r)
        mp, dyp, mask = _pad(m, ds, dr), _pad(dy, dr, dr), _pad(mask, ds, dr)
        dm = torch.empty_like(mp)
        outer_product_mean_backward(self.mod, mp.view(-1, C), mask[0], dyp.view(-1, Cz), None, dm.view(-1, C), g, s=s + ds, r=r + dr,
                                    nrm=F_.opm_normaliser(mask[0]), budget=self.budget)
        return dm[:, :s, :r].contiguous(), dy


def transition(tr, x):
    if not (as_built(tr) and covers_transition(tr) and _dtype_ok(x)):
        return None
    return _apply(_TransitionStep(tr), (x,), (), transition_parameters(tr))


def triangle_multiplication(tm, z, mask, drop):
    if not (as_built(tm) and covers_triangle_multiplication(tm) and _dtype_ok(z)):
        return None
    return _apply(_TriMulStep(tm), (z,), (mask, drop), triangle_multiplication_parameters(tm))


def triangle_attention(ta, z, mask, drop):
    if not (as_built(ta) and covers_triangle_attention(ta) and _dtype_ok(z)):
        return None
    return _apply(_TriAttStep(ta), (z,), (mask, drop), triangle_attention_parameters(ta))


def column_attention(col, m, mask):
    if not (as_built(col) and covers_column(col) and _dtype_ok(m)):
        return None
    return _apply(_ColumnStep(col), (m,), (mask,), column_parameters(col))


def row_attention(row, m, z, mask, drop):
    if not (as_built(row) and covers_row(row) and _dtype_ok(m, z)):
        return None
    return _apply(_RowStep(row), (m, z), (mask, drop), row_parameters(row))


def outer_product_mean(opm, m, mask, z, budget):
    if not (as_built(opm) and covers_outer_product_mean(opm) and _dtype_ok(m, z)) or m.dim() != 4:
        return None
    return _apply(_OuterStep(opm, budget), (m, z), (mask,), outer_product_mean_parameters(opm))


# ------------------------------------------------------------------------------------------------- block ----
def block_backward(block, m, z, msa_mask, pair_mask, dm, dz, dm_out, dz_out, g, drops, *, derived, budget):
    """m [1, s, r, c_m], z [1, r, r, c_z] (the block's inputs) and the cotangents of its outputs -> dm_out, dz_out and ``g``."""
    drops = drops or {}
    _, s, r, cm = m.shape
    cz = z.shape[-1]
    kb_row, kb_col, kb_start, kb_end, nrm = derived
    msa, pair, opm = block.msa, block.pair, block.communication

    def new(t):
        return alloc(tuple(t.shape), t.dtype, t.device)

    def dr(key, width):
        d = drops.get(key)
        return None if d is None else d.reshape(-1, width)
    # residual streams between the sub-modules, and two buffers of cotangents each
    m1, m2, m3 = new(m), new(m), new(m)
    z1, z2, z3, z4, z5 = (new(z) for _ in range(5))
    dza, dzb, dma, dmb = new(z), new(z), new(m), new(m)
    _plan.hold()
    mk, pk = msa_mask[0], pair_mask[0]
    multimer = block.is_multimer

    def outer(src):
        opm._run(src, msa_mask, z, z1)
    if multimer:
        outer(m)
    msa.MSARowAttentionWithPairBias._run(m, z1 if multimer else z, msa_mask, m1, drop=drops.get("row"))
    msa.MSAColumnAttention._run(m1, msa_mask, m2)
    if not multimer:
        msa.MSATransition._run(m2, m3)
        outer(m3)
    pair.TriangleMultiplicationOutgoing._run(z1, pair_mask, z2, drop=drops.get("tmo"))
    pair.TriangleMultiplicationIncoming._run(z2, pair_mask, z3, drop=drops.get("tmi"))
    pair.TriangleAttentionStartingNode._run(z3, pair_mask, z4, drop=drops.get("tas"))
    pair.TriangleAttentionEndingNode._run(z4, pair_mask, z5, drop=drops.get("tae"))

    def flat(t, c):
        return t.view(-1, c)
    Z, Mm = (lambda t: flat(t, cz)), (lambda t: flat(t, cm))

    def msa_back(dmo, zin, dzin, dm_to, dz_to):
        """Transition, column and row attention; the row attention's bias adds to ``dzin`` (in ``dz_to``)."""
        _plan.scope()
        transition_backward(msa.MSATransition, Mm(m2), Mm(dmo), Mm(dma), g)
        _plan.scope()
        col = msa.MSAColumnAttention
        attention_backward(col, col.attention, col.layernormM, Mm(m1), Mm(dma), Mm(dmb), g, col.attention.o_linear.bias, B2=r, N=s,
                           a_map=(s, cm, r * cm), kb=kb_col[0], flags=kb_col[1])
        _plan.scope()
        row_attention_backward(msa.MSARowAttentionWithPairBias, Mm(m), Z(zin), Mm(dmb), Mm(dm_to), Z(dzin), Z(dz_to), g,
                               s=s, r=r, kb=kb_row[0], flags=kb_row[1], drop=dr("row", cm))

    def pair_back(dzo):
        _plan.scope()
        transition_backward(pair.PairTransition, Z(z5), Z(dzo), Z(dza), g)
        src, dst = dza, dzb
        for ta, zin, a_map, kb, key, dmap in (
                (pair.TriangleAttentionEndingNode, z4, (r, cz, r * cz), kb_end, "tae", (r, cz, 0)),
                (pair.TriangleAttentionStartingNode, z3, (r * r, 0, cz), kb_start, "tas", (r, 0, cz))):
            _plan.scope()
            attention_backward(ta, ta.attention, ta.layernorm1, Z(zin), Z(src), Z(dst), g, ta.out_bias, B2=r, N=r, a_map=a_map,
                               kb=kb[0], flags=kb[1], linear_b=ta.linear_b, drop=dr(key, cz), drop_map=dmap)
            src, dst = dst, src
        for tm, zin, key in ((pair.TriangleMultiplicationIncoming, z2, "tmi"), (pair.TriangleMultiplicationOutgoing, z1, "tmo")):
            _plan.scope()
            triangle_multiplication_backward(tm, Z(zin), Z(src), Z(dst), g, r=r, mask=pk, drop=dr(key, cz))
            src, dst = dst, src
        return src

    def outer_back(src, dzo, dm_in, dm_to):
        _plan.scope()
        outer_product_mean_backward(opm, Mm(src), mk, Z(dzo), None if dm_in is None else Mm(dm_in), Mm(dm_to), g, s=s, r=r, nrm=nrm,
                                    budget=budget)
    dz1 = pair_back(dz)
    if multimer:
        # the MSA stack read z1, and m went into the outer product as well
        msa_back(dm, z1, dz1, dma, dz_out)
        outer_back(m, dz_out, dma, dm_out)
    else:
        outer_back(m3, dz1, dm, dmb)
        msa_back(dmb, z, dz1, dm_out, dz_out)
