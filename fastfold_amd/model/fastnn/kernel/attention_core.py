"""``fused_attention_core`` with the reference's interface
(fastfold/model/fastnn/kernel/attention_core.py:17-52):

    softmax(q * d**-0.5 @ k^T + bias + BIG * (mask - 1)) @ v   ->   [b1, b2, n, h*d]

for q, k, v ``[b1, b2, h, n, d]``, mask ``[b1, b2, n]`` (0/1, over keys) and bias ``[b1, h, n, n]``.
The logits are never materialised: the operands are re-tiled into the 32x32 MFMA order and handed to
the flash attention kernel (``ffk_attention_fwd``, ``ffk_attention_fwd_lse``); the backward pass (``ffk_attention_bwd_rows``, for
wide heads ``ffk_attention_bwd``) recomputes them the same way.  The tuned kernel is the Evoformer's head dim (32); narrower heads (8 and 16, the extra-MSA and template
stacks) are zero-padded to 32 channels, which changes neither the scores nor the used output channels; the other
widths the reference's Triton kernel takes (64 and 128, triton/attention_core.py:142), which no module of the path
uses, run on a plain one-wave-per-query-tile instantiation that cuts the head into 32-channel parts.
Dtypes: bf16 and fp32 (forward and backward); fp16 raises here, before anything is launched.
"""
import math

import torch

from .... import _lib
from . import layouts


def _check(q, k, v, mask, bias):
    for t in (q, k, v, mask, bias):          # any strides: the operands are re-tiled as they lie
        if t is not None and not t.is_cuda:
            raise RuntimeError("fastfold_amd: tensor must be a CUDA/HIP tensor (got %s)" % t.device)
    if q.dim() != 5 or q.shape != k.shape or q.shape != v.shape:
        raise RuntimeError("fused_attention_core: q, k, v must be [b1, b2, h, n, d] of one shape, got %s %s %s"
                           % (tuple(q.shape), tuple(k.shape), tuple(v.shape)))
    b1, b2, h, n, d = q.shape
    if d not in (8, 16, 32, 64, 128):
        raise RuntimeError("fused_attention_core: head dim %d is not supported (8, 16, 32, 64 or 128)" % d)
    if q.dtype not in (torch.bfloat16, torch.float32) or k.dtype != q.dtype or v.dtype != q.dtype:
        raise RuntimeError("fused_attention_core: q, k, v must share one dtype, bfloat16 or float32 (got %s, %s, %s)"
                           % (q.dtype, k.dtype, v.dtype))
    if mask is not None and tuple(mask.shape) != (b1, b2, n):
        raise RuntimeError("fused_attention_core: mask must be [b1, b2, n], got %s" % (tuple(mask.shape),))
    if bias is not None and tuple(bias.shape) != (b1, h, n, n):
        raise RuntimeError("fused_attention_core: bias must be [b1, h, n, n], got %s" % (tuple(bias.shape),))


def _key_bias(kb, fl, mask, b2, n, dt, dev):
    mk = mask.to(dt).contiguous() if mask is not None else torch.ones(b2, n, dtype=dt, device=dev)
    _lib.key_bias(kb, fl, mk, B=b2, N=n, mask_sb=n, mask_sn=1)


def _attention_core_wide(q, k, v, mask, bias):
    """Head dims 64 and 128."""
    b1, b2, h, n, d = q.shape
    out = torch.empty(b1, b2, n, h * d, dtype=q.dtype, device=q.device)
    nt = layouts.n_tiles(n)
    kb = torch.empty(b2, nt * 32, dtype=torch.float32, device=q.device)
    fl = torch.empty(b2, nt, dtype=torch.int32, device=q.device)
    for i in range(b1):
        _key_bias(kb, fl, None if mask is None else mask[i], b2, n, q.dtype, q.device)
        bt = layouts.tile_bias((bias[i].float() * _lib.LOG2E).to(q.dtype)) if bias is not None else None
        _lib.attention_fwd(out[i].view(b2 * n, h * d), _lib.tile_pack(q[i], _lib.FFK_TILE_QK, _lib.LOG2E / math.sqrt(d)),
                           _lib.tile_pack(k[i], _lib.FFK_TILE_QK), _lib.tile_pack(v[i], _lib.FFK_TILE_V), bt, kb, fl,
                           None, B2=b2, H=h, Nq=n, Nk=n, D=d)
    return out


def _at(t, i):
    """Address and strides of element i of the first of the five dimensions of t."""
    sb, *rest, _ = t.stride()
    return (t.data_ptr() + i * sb * t.element_size(), *rest)


def _attention_core(q, k, v, mask=None, bias=None, keep=False):
    """Head dims 8, 16 and 32.  ``keep``: also what the backward pass reads - the q and k tiles, the rows' log-sum-exp, the key
    bias of the mask and the bias tiles, one set per b1."""
    b1, b2, h, n, d = q.shape
    dt, dev = q.dtype, q.device
    nt = layouts.n_tiles(n)
    # zero channels past d add nothing to q.k and give zero output channels, which are dropped at the end
    out = torch.empty(b1, b2, n, h * 32, dtype=dt, device=dev)
    kept = b1 if keep else 1
    qk = torch.empty(kept, 2, b2, h, nt, 1024, dtype=dt, device=dev)
    vt = torch.empty(b2, h, nt, 1024, dtype=dt, device=dev)
    bt = torch.empty(kept, h, nt, nt, 1024, dtype=dt, device=dev) if bias is not None else None
    kb = torch.empty(kept, b2, nt * 32, dtype=torch.float32, device=dev)
    fl = torch.empty(b2, nt, dtype=torch.int32, device=dev)
    lse = torch.empty(b1, b2 * h * nt * 32, dtype=torch.float32, device=dev) if keep else None
    q, k, v = (t if t.stride(-1) == 1 else t.contiguous() for t in (q, k, v))
    mask = mask.to(dt).contiguous() if mask is not None else torch.ones(1, b2, n, dtype=dt, device=dev).expand(b1, b2, n)
    bscale = 1.0
    if bias is not None:                      # the kernel exponentiates in base 2
        bias, bscale = ((bias.contiguous(), _lib.LOG2E) if bias.dtype == dt else ((bias.float() * _lib.LOG2E).to(dt).contiguous(), 1.0))
    # addresses instead of views: a view of a tensor costs the host as much as a launch
    es, tiles = q.element_size(), b2 * h * nt * 1024 * q.element_size()
    for i in range(b1):
        s = i if keep else 0
        qt = qk.data_ptr() + 2 * s * tiles
        kbi = kb.data_ptr() + s * b2 * nt * 128
        bti = None if bt is None else bt.data_ptr() + s * h * nt * nt * 1024 * es
        _lib.call("ffk_key_bias", kbi, fl.data_ptr(), mask.data_ptr() + i * mask.stride(0) * es, b2, n, n, 1, _lib.dtype_tag(dt),
                  _lib.stream_ptr())
        _lib.attention_pack([(_at(q, i), _lib.LOG2E / math.sqrt(d), qt, None, None, None), (_at(k, i), 1.0, qt + tiles, None, None, None),
                             (_at(v, i), 1.0, None, vt, None, None)],
                            B2=b2, H=h, N=n, D=d, dtype=dt, bias=None if bt is None else bias.data_ptr() + i * h * n * n * es, bias_t=bti,
                            bias_scale=bscale)
        _lib.attention_fwd_lse(out.data_ptr() + i * b2 * n * h * 32 * es, None if lse is None else lse.data_ptr() + i * b2 * h * nt * 128,
                               qt, qt + tiles, vt, bti, kbi, fl, B2=b2, H=h, N=n, dtype=dt)
    if d < 32:
        out = out.view(b1, b2, n, h, 32)[..., :d].reshape(b1, b2, n, h * d)
    return (out, qk, kb, bt, lse) if keep else out


def _attention_core_backward(qk, v, kb, bt, lse, out, dout, need_dbias):
    """dq, dk, dv (shape of v) and dbias ([b1, h, n, n] or None) for head dims up to 32, from what the forward pass kept."""
    b1, b2, h, n, d = v.shape
    dt, dev = v.dtype, v.device
    nt = layouts.n_tiles(n)
    dq, dk, dv = (torch.empty(b1, b2, h, n, 32, dtype=dt, device=dev) for _ in range(3))
    es, tiles = v.element_size(), b2 * h * nt * 1024 * v.element_size()
    work = torch.empty(5, b2, h, nt, 1024, dtype=dt, device=dev)
    q_acc, k_acc, v_qk, do_qk, do_acc = (work.data_ptr() + j * tiles for j in range(5))
    dsum = torch.empty(b2 * h * nt * 32, dtype=torch.float32, device=dev)
    parts, dbias = 0, None
    if need_dbias and bt is not None:
        # partial sums over slices of the batch rows, at least eight each: the four waves per SIMD that are resident together
        parts = max(1, min(-(-4096 // (h * nt * nt)), (b2 + 7) // 8))
        part = torch.empty(parts, h, n, n, dtype=torch.float32, device=dev)
        dbias = torch.empty(b1, h, n, n, dtype=dt, device=dev)
    v = v if v.stride(-1) == 1 else v.contiguous()
    rows = (n * h * d, d, h * d)                                     # strides of dout and out as [b2, h, n, d]
    for i in range(b1):
        qt = qk.data_ptr() + 2 * i * tiles
        off, grad = i * b2 * n * h * d * es, i * b2 * h * n * 32 * es
        _lib.attention_pack([((qt,), 1.0, None, q_acc, None, None), ((qt + tiles,), 1.0, None, k_acc, None, None),
                             (_at(v, i), 1.0, v_qk, None, None, None),
                             ((dout.data_ptr() + off, *rows), 1.0, do_qk, do_acc, dsum, (out.data_ptr() + off, *rows))],
                            B2=b2, H=h, N=n, D=d, dtype=dt)
        _lib.attention_bwd_rows(dq.data_ptr() + grad, dk.data_ptr() + grad, dv.data_ptr() + grad, part if parts else None,
                                lse.data_ptr() + i * b2 * h * nt * 128, dsum, qt, q_acc, qt + tiles, k_acc, v_qk,
                                None if bt is None else bt.data_ptr() + i * h * nt * nt * 1024 * es, kb.data_ptr() + i * b2 * nt * 128,
                                do_qk, do_acc, B2=b2, H=h, N=n, s_b=h * n * 32, s_h=n * 32,
                                s_n=32, dq_scale=1.0 / math.sqrt(d), dk_scale=1.0 / _lib.LOG2E, dtype=dt, dbias_parts=parts)
        if parts and h * n * n % 4 == 0:
            _lib.slice_sum(dbias[i], part, slices=parts, N=1, K=h * n * n, o_map=(1, 0, 0, 1), dtype=dt)
        elif parts:
            torch.sum(part, 0, out=dbias[i]) if dt == torch.float32 else dbias[i].copy_(part.sum(0))
    if d < 32:
        dq, dk, dv = (t[..., :d] for t in (dq, dk, dv))
    return dq, dk, dv, dbias


def _attention_core_backward_wide(q, k, v, mask, bias, out, dout, need_dbias):
    """The same for head dims 64 and 128, through ``ffk_attention_bwd``."""
    b1, b2, h, n, d = q.shape
    dt, dev = q.dtype, q.device
    QK, ACC = _lib.FFK_TILE_QK, _lib.FFK_TILE_V
    nt = layouts.n_tiles(n)
    scale = _lib.LOG2E / math.sqrt(d)
    dq, dk, dv = (torch.empty(b1, b2, h, n, d, dtype=dt, device=dev) for _ in range(3))
    dbias = torch.zeros(b1, h, n, n, dtype=torch.float32, device=dev) if (need_dbias and bias is not None) else None
    kb = torch.empty(b2, nt * 32, dtype=torch.float32, device=dev)
    fl = torch.empty(b2, nt, dtype=torch.int32, device=dev)
    lse = torch.empty(b2 * h * nt * 32, dtype=torch.float32, device=dev)
    dsum = torch.empty_like(lse)
    for i in range(b1):
        _key_bias(kb, fl, None if mask is None else mask[i], b2, n, dt, dev)
        bt = layouts.tile_bias((bias[i].float() * _lib.LOG2E).to(dt)) if bias is not None else None
        do_ = dout[i].view(b2, n, h, d).permute(0, 2, 1, 3)          # [b2, h, n, d] views: re-tiled as they lie
        o_ = out[i].view(b2, n, h, d).permute(0, 2, 1, 3)
        _lib.attention_bwd(dq[i], dk[i], dv[i], None if dbias is None else dbias[i], lse, dsum,
                           _lib.tile_pack(q[i], QK, scale), _lib.tile_pack(q[i], ACC, scale),     # as the forward saw q
                           _lib.tile_pack(k[i], QK), _lib.tile_pack(k[i], ACC), _lib.tile_pack(v[i], QK),
                           bt, kb,
                           _lib.tile_pack(do_, QK), _lib.tile_pack(do_, ACC), _lib.tile_pack(o_, QK),
                           B2=b2, H=h, Nq=n, Nk=n, D=d, dq_scale=1.0 / math.sqrt(d), dk_scale=1.0 / _lib.LOG2E)
    return dq, dk, dv, (None if dbias is None else dbias.to(dt))


class FusedAttenionCoreFunc(torch.autograd.Function):
    """Name (including its spelling) as in the reference (attention_core.py:34).  The reference's function has no
    backward (training goes through matmul / fused_softmax / matmul there, fastnn/ops.py:310-322); this one has:
    dq, dk, dv and dbias from ``ffk_attention_bwd_rows`` and ``ffk_attention_bwd``, which recompute the logits tile by tile."""

    @staticmethod
    def forward(ctx, q, k, v, mask=None, bias=None):
        _check(q, k, v, mask, bias)
        grads = any(t is not None and t.requires_grad for t in (q, k, v, bias))
        b1, b2, h, n, d = q.shape
        ctx.wide = d > 32
        ctx.empty = q.numel() == 0
        if ctx.empty:
            ctx.save_for_backward(q, k, v, bias)
            return torch.empty(b1, b2, n, h * d, dtype=q.dtype, device=q.device)
        if ctx.wide:
            out = _attention_core_wide(q, k, v, mask, bias)
            if grads:
                ctx.save_for_backward(q, k, v, mask, bias, out)
        elif grads:
            out, qk, kb, bt, lse = _attention_core(q, k, v, mask, bias, keep=True)
            ctx.save_for_backward(qk, v, kb, bt, lse, out)
        else:
            out = _attention_core(q, k, v, mask, bias)
        return out

    @staticmethod
    def backward(ctx, dout):
        if ctx.empty:
            dq, dk, dv, dbias = (None if t is None else torch.zeros_like(t) for t in ctx.saved_tensors)
            return dq, dk, dv, None, dbias
        back = _attention_core_backward_wide if ctx.wide else _attention_core_backward
        saved = ctx.saved_tensors
        dq, dk, dv, dbias = back(*saved[:-1], saved[-1].contiguous(), dout.contiguous(), ctx.needs_input_grad[4])
        return dq, dk, dv, None, dbias


fused_attention_core = FusedAttenionCoreFunc.apply
