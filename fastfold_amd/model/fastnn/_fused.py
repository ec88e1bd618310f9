"""Launch sequences of the HIP kernels for each Evoformer sub-module (single GPU, DAP size 1).

These functions take plain tensors plus weights already packed for the kernels and issue
C-ABI calls only; torch is used for buffer allocation and for re-packing weights (once per
weight version).  Row-addressing conventions are those of ``ffk_fused_linear``: logical row
``m = hi * inner + lo`` lives at ``hi * s_o + lo * s_i``.
"""
import contextlib
import math
import os
import threading

import torch

from fastfold_amd import _lib, _plan
from fastfold_amd._lib import (FFK_ACT_NONE, FFK_ACT_RELU, FFK_ACT_SIGMOID, FFK_TILE_ACC, FFK_TILE_BIAS, FFK_TILE_QK,
                               FFK_TILE_STRIDED, FFK_TILE_V, LOG2E, make_tile)

_WS_BUDGET_DEFAULT = 6 << 30     # bytes of scratch one sub-module may hold at a time
_WS_BUDGET_CHUNKED = 1 << 30     # when the user asked for chunking (set_chunk_size)


def es_of(dtype):
    return 4 if dtype == torch.float32 else 2


def vec_of(dtype):
    return 16 // es_of(dtype)


def round_up(x, m):
    return (x + m - 1) // m * m


def alloc(shape, dtype, device, zero=False):
    """A scratch tensor of the launch sequences below."""
    t = _plan.alloc(torch.empty(shape, dtype=dtype, device=device))
    if zero:
        if t.numel() * t.element_size() % 16:
            raise RuntimeError("alloc: zeroed scratch must be a multiple of 16 bytes, got %s" % (tuple(t.shape),))
        _lib.fill_zero(t)
    return t


def switches():
    """Everything besides shapes and dtypes that the launch sequences below depend on."""
    return (_WS_BUDGET_DEFAULT, _WS_BUDGET_CHUNKED, _FUSED_TRANSITION, _TRIMUL_CHAN_PAD, _PAIR_BIAS_RIDES, _BIAS_ROW_PAD,
            _GATE_IN_OUT_STAGE, _GATE_IN_OUT_MIN_N, _GATE_IN_OUT_WIDTHS, _ATTENTION_BLOCK)


def pack_rows(mats, dtype, device):
    """cat([n_i, K]) zero-padded to a multiple of 128 rows, in the kernel dtype."""
    w = torch.cat([m.detach().to(device=device, dtype=dtype) for m in mats], 0)
    n, npad = w.shape[0], round_up(w.shape[0], 128)
    if npad != n:
        w = torch.cat([w, w.new_zeros(npad - n, w.shape[1])], 0)
    return w.contiguous()


def pack_vec(vecs, dtype, device, total=None):
    v = torch.cat([x.detach().to(device=device, dtype=dtype).reshape(-1) for x in vecs], 0)
    total = round_up(v.numel(), 128) if total is None else total
    if total != v.numel():
        v = torch.cat([v, v.new_zeros(total - v.numel())], 0)
    return v.contiguous()


def check_cuda(*ts):
    for t in ts:
        if t is not None and not t.is_cuda:
            raise RuntimeError("fastfold_amd: the Evoformer modules run on the GPU only "
                               "(got a %s tensor); there is no CPU fallback" % t.device)


def check_nonempty(who, *ts):
    """The kernels take at least one sequence and one residue; an empty tensor is an error of the caller."""
    for t in ts:
        if t is not None and t.numel() == 0:
            raise RuntimeError("%s: empty input tensor of shape %s" % (who, tuple(t.shape)))


# ---- values derived from a mask only (key bias + tile flags of an attention, the normaliser of the outer
# product mean) are the same in every block of a stack: inside `mask_cache()` they are computed once ----
class _MaskCache(threading.local):
    entries = None           # of the calling thread, while in a mask_cache()


_MASK_CACHE = _MaskCache()


def mask_scope():
    """The running ``mask_cache``, or one for the caller's block alone."""
    return mask_cache() if _MASK_CACHE.entries is None else contextlib.nullcontext()


@contextlib.contextmanager
def mask_cache():
    """While active, launches whose result depends only on a mask tensor are done once per distinct
    (storage, view geometry, version) and reused.  Entries keep their mask alive, so its memory cannot be
    handed to another tensor while the entry exists; the cache dies with the context."""
    prev, _MASK_CACHE.entries = _MASK_CACHE.entries, []
    try:
        yield
    finally:
        _MASK_CACHE.entries = prev


def _mask_derived(mask, what, build):
    entries = _MASK_CACHE.entries
    if entries is None:
        return build()
    # tensors made under torch.inference_mode have no version counter; a cache lives within one call of a stack or block,
    # during which nobody writes the masks it was given
    version = None if mask.is_inference() else mask._version
    key = (what, mask.data_ptr(), version, tuple(mask.shape), tuple(mask.stride()), mask.dtype)
    for k, _, v in entries:
        if k == key:
            return v
    v = build()
    if len(entries) < 32:              # a stack needs about ten; bounded whatever the caller does
        entries.append((key, mask, v))
    return v


class PairBiasScratch:
    """Device scratch of ffk_pair_bias together with the fact that it already holds the weight operand
    (built by the first call from the projection weights and the LayerNorm parameters); modules keep one
    per packed weight set, so that later calls skip the preparation kernel."""

    def __init__(self, C, device):
        self.buf = torch.empty(16 * C + 16, dtype=torch.float32, device=device)
        self.ready = False


def _pair_bias_launch(bias_t, x, ln, w, scratch, **kw):
    if scratch is None:
        scratch = PairBiasScratch(x.shape[-1], x.device)
    if not scratch.ready:
        _plan.note_build()
    _lib.pair_bias(bias_t, x, ln[0], ln[1], None if scratch.ready else w, scratch.buf, **kw)
    scratch.ready = True


def aligned16(*ts):
    """Whether 16-byte loads may read the tensors from their first element.  Parameters come as they are (slices of a flat buffer, say);
    the kernels that need whole vectors of them are taken only then."""
    return all(t.data_ptr() % 16 == 0 for t in ts)


def fits_fused(K, dtype):
    return K <= 256 and K % 32 == 0


def pad_to_tiles(m, z, msa_mask, pair_mask, pad_s=True):
    """m [1, s, r, c_m], z [1, r, r, c_z] and their masks, zero-padded to whole 32-row tiles along the residue axis and
    (``pad_s``) the sequence axis; bf16 tensors whose extents are no multiples of 32, everything else as it came.

    The padding is masked: no un-padded result reads it.  It exists because the fast kernels work on whole tiles: the
    weights-stationary projections write attention operands in accumulator order for rows of whole 32-key tiles, the
    triangle multiplication's output stage and the fused outer product want r % 8 == 0 and r % 32 == 0.  The rows added
    (at most 31 of each axis: 13 % of the pair positions at 391 residues) cost less than the LDS-staged kernels a ragged
    extent would take at every size measured: 8 blocks at N_seq = 125, N_res = 391 18.1 -> 10.9 ms.  fp32 runs on the
    staged kernels at any extent, so padding would only add work there.

    In-place calls pad too.  The copies lie beside the caller's tensors, but the un-padded run held as much in gate tensors and
    unfused scratch: one block in place at N_seq = 64, N_res = 4 090, bytes beyond the inputs and time, padded 19.8 GB and
    208 ms, un-padded 19.6 GB and 296 ms; at 1 270 2.0 GB and 11.3 ms, 1.9 GB and 19.4 ms.  (4 096, without copies: 15.3 GB.)"""
    s, r = m.shape[1], m.shape[2]
    if m.dtype != torch.bfloat16:
        return m, z, msa_mask, pair_mask
    ds, dr = (round_up(s, 32) - s if pad_s else 0), round_up(r, 32) - r
    if ds == 0 and dr == 0:
        return m, z, msa_mask, pair_mask
    pad = torch.nn.functional.pad
    if dr:
        z, pair_mask = pad(z, (0, 0, 0, dr, 0, dr)), pad(pair_mask, (0, dr, 0, dr))
    return pad(m, (0, 0, 0, dr, 0, ds)), z, pad(msa_mask, (0, dr, 0, ds)), pair_mask


# ------------------------------------------------------------------------- linear ----
def linear(x2, w_pk, b_pk, N, *, act=FFK_ACT_NONE, out=None, resid=None, ln=None):
    """out[M, N] = act(LN(x2)[M, K] @ W^T + b) (+ resid).  ``w_pk`` is [>=N (padded to 128), K]."""
    M, K = x2.shape
    dt, dev = x2.dtype, x2.device
    es = es_of(dt)
    if out is None:
        out = torch.empty(M, N, dtype=dt, device=dev)
    if M == 0:
        return out
    if fits_fused(K, dt) and N % vec_of(dt) == 0:
        nt = (N + 127) // 128
        for t0 in range(0, nt, _lib.FFK_MAX_TILES):
            tiles = []
            for t in range(t0, min(nt, t0 + _lib.FFK_MAX_TILES)):
                tiles.append(make_tile(out.data_ptr() + t * 128 * es,
                                       bias=None if b_pk is None else b_pk.data_ptr() + t * 128 * es,
                                       resid=None if resid is None else resid.data_ptr() + t * 128 * es,
                                       inner=M, s_i=N, act=act, ncols=min(128, N - t * 128)))
            _lib.fused_linear(x2, w_pk, tiles, M=M, K=K, ln=ln, w_row_off=t0 * 128)
    else:
        if ln is not None:
            raise RuntimeError("linear: LayerNorm prologue needs K <= 256")
        if K % vec_of(dt) != 0:
            raise RuntimeError("linear: in_features=%d must be a multiple of %d for %s" % (K, vec_of(dt), dt))
        _lib.bgemm_nt(x2, w_pk, out, M=M, N=N, K=K, lda=K, ldb=K, bias=b_pk, resid=resid, act=act)
    return out


# --------------------------------------------------------------------- transition ----
def xtail_ptr(xtail, off=0):
    """Address of element ``off`` of an int8 residual tail (None stays None)."""
    return None if xtail is None else xtail.data_ptr() + off


# False: every transition runs as projection + GEMM with the hidden activation in HBM (tests compare the two)
_FUSED_TRANSITION = True


def transition_block_rows(C):
    """Most rows ``ffk_transition_block`` is taken for (timings of both sides in csrc/ffk_transition_block.hip).  The kernel behind the line
    gives the same bits: a rank's share of the rows, or a piece of them, gets those of the full call."""
    return 16384 if C == 128 else 1 << 36


def transition_takes_block(M, C, w_block, ln, b2):
    return w_block is not None and ln is not None and _FUSED_TRANSITION and M <= transition_block_rows(C) and aligned16(*ln, b2)


def transition(x, out, *, ln, w1_pk, b1_pk, w2, b2, hidden, budget, xtail=None, w_block=None):
    """out = x + W2 relu(W1 LN(x) + b1) + b2 over rows of x [M, C]; out may alias x.  ``w_block``: the weights as
    ``pack_transition_block`` lays them out, or None; ``w1_pk`` is needed where ``transition_takes_block`` is false.  ``xtail`` (here and in the
    other sub-modules): int8 tensor of x's shape holding the tail bytes of x / out as an extended residual stream."""
    M, C = x.shape
    dt, dev = x.dtype, x.device
    es = es_of(dt)
    if transition_takes_block(M, C, w_block, ln, b2):
        _lib.transition_block(out, x, ln[0], ln[1], w_block[0], b1_pk, w_block[1], b2, M=M, C=C, hidden=hidden, xtail=xtail)
        return out
    if dt == torch.bfloat16 and C in (128, 256) and hidden == 4 * C and ln is not None and _FUSED_TRANSITION:
        # both layers in one kernel, hidden activation kept on chip: many rows of 128 channels (256: ffk_transition_block takes all but
        # parameters that are not aligned, which this kernel does not take either)
        _lib.transition_fused(out, x, ln[0], ln[1], w1_pk, b1_pk, w2, b2, M=M, C=C, hidden=hidden, xtail=xtail)
        return out
    rows = max(128, min(M, (budget // (hidden * es)) // 128 * 128))
    hid = alloc((min(rows, M), hidden), dt, dev)
    nt = hidden // 128
    for r0 in range(0, M, rows):
        n = min(rows, M - r0)
        per = _lib.WS_TILES if dt == torch.bfloat16 else _lib.FFK_MAX_TILES
        for t0 in range(0, nt, per):
            tiles = [make_tile(hid.data_ptr() + t * 128 * es, bias=b1_pk.data_ptr() + t * 128 * es, inner=n,
                               s_i=hidden, act=FFK_ACT_RELU)
                     for t in range(t0, min(nt, t0 + per))]
            _lib.fused_linear(x, w1_pk, tiles, M=n, K=C, ln=ln, a_off=r0 * C, w_row_off=t0 * 128)
        _lib.bgemm_nt(hid, w2, out.data_ptr() + r0 * C * es, M=n, N=C, K=hidden, lda=hidden, ldb=hidden, bias=b2,
                      resid=x.data_ptr() + r0 * C * es, dtype=dt, xtail=xtail_ptr(xtail, r0 * C))
    return out


# ---------------------------------------------------------------------- attention ----
def key_bias(mask, device, *, B2, N, mask_sb, mask_sn):
    """(additive key bias, key-tile flags) of an attention over B2 rows of N keys; from a mask once per ``mask_cache``."""
    def build():
        NT = (N + 31) // 32
        kb = torch.empty(B2, NT * 32, dtype=torch.float32, device=device)
        flags = torch.empty(B2, NT, dtype=torch.int32, device=device)
        _lib.key_bias(kb, flags, mask, B=B2, N=N, mask_sb=mask_sb, mask_sn=mask_sn)
        return kb, flags
    return build() if mask is None else _mask_derived(mask, ("key_bias", B2, N, mask_sb, mask_sn), build)


def attention_block_tokens(dtype, H, c, d_in, d_out):
    """Longest row of tokens that ``ffk_attention_block`` takes at these widths, 0 where it is not built for them.

    Rows go to it by their length and width only, never by how many there are: a subset of the batch rows must give the bits of the
    full call.  One row keeps a CU busy whatever the others do, so it loses where few long rows leave CUs idle or the last round of
    rows is nearly empty.  us per sub-module, one kernel / launches of their own:
      128 channels in heads of 32, N rows of N tokens: 32 13.4 / 14.0, 96 19.3 / 24.5, 160 28 / 43, 224 42 / 64, 256 49 / 67
      64 channels in heads of 16, the same: 64 11.0 / 18.5, 256 31 / 52, 288 68 / 71, 320 76 / 83, 352 92 / 94, 384 98 / 104, 512 161 / 191
      64 channels in heads of 8, 64 / 256 / 384 / 1 024 rows: 96 tokens 18 / 22, 19 / 36, 30 / 47, 54 / 79; 160 31 / 29, 32 / 55, 53 / 70,
        99 / 150; 256 46 / 34, 49 / 69, 86 / 91, 163 / 205; 384 92 / 47, 96 / 114, 170 / 154, 327 / 397 (of the 64 rows that a stack of
        extra sequences hardly has, more than 192 tokens lose; from 192 rows on all lengths win but at 384 rows)
      256 channels without a bias, 32 / 64 / 256 / 1 024 rows: 64 tokens 14 / 19, 15 / 23, 18 / 47, 66 / 132; 96 20.5 / 21.8, 21 / 31, 27 / 61,
        101 / 213; 128 27.5 / 24.0, 28 / 34, 34 / 72, 126 / 276
      256 channels with one, 32 / 64 / 128 / 512 rows: 96 tokens 27 / 28, 27 / 37, 28 / 47, 61 / 106; 128 35 / 31, 35 / 39, 36 / 55, 77 / 135
      the heads apart (``ATTENTION_HEADS_TOKENS``), 32 / 64 / 128 / 160 / 512 rows: 160 tokens 36.7 / 36.8, 42 / 48, 49 / 68, 71 / 82, 142 / 190;
        192 42 / 38, 47 / 50, 54 / 75, 80 / 87, 164 / 233; 224 51 / 39, 55 / 56, 66 / 85, 99 / 100, 203 / 271; 256 57 / 40, 61 / 58, 73 / 89,
        110 / 104, 232 / 303"""
    if dtype != torch.bfloat16 or d_in != d_out or H * c != d_in:
        return 0
    return {(128, 32): 256, (64, 16): 512, (64, 8): 384, (256, 32): 128}.get((d_in, c), 0)


def pack_attention_block(qkv_w, gate_w, out_w, dtype, device):
    """The weights of a gated attention in the fragment order of ``ffk_attention_block``: [q, k, v, gate, out][C/32][C/16][64][8]."""
    w = torch.empty(qkv_w.numel() + gate_w.numel() + out_w.numel(), dtype=dtype, device=device)
    at = 0
    for part in (fragments(qkv_w), fragments(gate_w), fragments_of_accumulators(out_w)):       # one launch each
        w[at:at + part.numel()].view(part.shape).copy_(part)
        at += part.numel()
    return w


def fragments(w):
    """[n, K] as [n/32][K/16][half][row][8]: what each lane of a wave gives to the matrix instructions that multiply by 32 rows of w."""
    w = w.detach()
    return w.reshape(w.shape[0] // 32, 32, w.shape[1] // 16, 2, 8).permute(0, 2, 3, 1, 4)


def fragments_of_accumulators(w):
    """The same for a weight that multiplies accumulators as they stand: columns in their order ([quad][half][4] of a step), and rows
    (8 a + 4 h + b from 16 h + 4 a + b) so that a lane's results are 16 consecutive channels."""
    w = w.detach()
    return w.reshape(w.shape[0] // 32, 2, 4, 4, w.shape[1] // 16, 2, 2, 4).permute(0, 4, 6, 2, 1, 3, 5, 7)


def pack_fragments(w, dtype, device):
    return fragments(w).to(device=device, dtype=dtype).reshape(-1)


def pack_fragments_of_accumulators(w, dtype, device):
    return fragments_of_accumulators(w).to(device=device, dtype=dtype).reshape(-1)


ATTENTION_HEADS_TOKENS = 256     # longest row of ffk_attention_heads


def pack_transition_block(w1, w2, dtype, device):
    """The weights of a transition in the fragment order of ``ffk_transition_block``; None at widths it is not built for."""
    hidden, C = w1.shape
    if dtype != torch.bfloat16 or (C, hidden) not in ((64, 128), (64, 256), (128, 512), (256, 1024)):
        return None
    w1, w2 = w1.detach(), w2.detach()
    # rows of w1 in the order (16 a + 8 c + 4 h + b from 16 a + 8 h + 4 c + b) in which a lane's sums are consecutive hidden channels,
    # the second layer's operand in the order of ffk_transition_fused; rows of w2 as in fragments_of_accumulators
    f1 = w1.reshape(hidden // 32, 2, 2, 2, 4, C // 16, 2, 8).permute(0, 5, 6, 1, 3, 2, 4, 7)
    f2 = w2.reshape(C // 32, 2, 4, 4, hidden // 16, 2, 8).permute(0, 4, 5, 2, 1, 3, 6)
    return tuple(f.to(device=device, dtype=dtype).reshape(-1) for f in (f1, f2))


# False: every attention runs as projection, core and output stage (tests compare the two)
_ATTENTION_BLOCK = True


def attention(x, out, resid, *, B2, N, C, H, a_map, ln, w_pk, gate_bias_pk, wo_pk, out_bias_pk, c_out,
              mask, mask_sb, mask_sn, bias_t=None, bias_in_launch=False, pb_scratch=None, head_dim=32, budget=None, o_map=None, xtail=None,
              drop=None):
    """Gated multi-head attention over N tokens for each of B2 batch rows.  The kernels work on 32-channel tiles.  Heads of
    8 or 16 channels lie side by side in them (``w_pk.packed_heads``) where the operands are written in accumulator order;
    elsewhere, and at other widths, a narrower head (``head_dim`` < 32) arrives zero-padded to 32 channels in ``w_pk`` / ``wo_pk``,
    which changes neither the scores nor the used output channels - only the score scale is its own.

    x holds the C-channel rows addressed by ``a_map = (inner, s_o, s_i)`` with ``inner`` either B2 * N (plain
    row-major) or N (one batch row per outer step); w_pk is the packed [q; k; v; gate(; bias)] weight.  The
    attention update is projected by wo_pk and written as ``out = resid + update + out_bias`` with the same row
    addressing, or with ``o_map`` if the output rows have another width (``resid=None``: no residual).  With ``bias_in_launch`` the last N-tile of w_pk produces the
    [H, N, N] additive bias into ``bias_t`` from the same normalised rows.

    ``budget`` (bytes) bounds the operand buffers (q, k, v, gate and the head outputs: 5 * H * ceil(N / 32) KB
    elements per batch row): the batch rows are then processed in slabs - projection, core, output projection per
    slab.  Batch rows are independent and a slab's outputs overwrite only the rows it read, so this also holds
    when ``out`` aliases ``x``; the additive bias, which reads all of x, is computed before the first slab.

    ``drop``: None, or a [period, c_out] tensor of dropout multipliers (0 or 1 / (1 - p)) that scales the update of logical
    row m by its row ``m % period`` before the residual is added (the shared-axis dropout of the training mode:
    ``bias_dropout_add`` with a mask drawn by the caller).
    """
    dt, dev = x.dtype, x.device
    es = es_of(dt)
    M = B2 * N
    NT = (N + 31) // 32
    zero = (N % 32) != 0
    a_inner, a_so, a_si = a_map
    o_inner, o_so, o_si = a_map if o_map is None else o_map
    if a_inner not in (M, N) or o_inner != a_inner:
        raise RuntimeError("attention: row maps with inner=%d / %d fit neither B2 * N nor N" % (a_inner, o_inner))
    # With bf16, 128 input channels and whole key tiles the projection runs on the weights-stationary
    # kernel, which writes q, k and the gate in accumulator order straight from its registers.
    acc_order = dt == torch.bfloat16 and C in (64, 128, 256) and N % 32 == 0
    # Short rows: one kernel from the rows of x to the updated rows.
    short = _ATTENTION_BLOCK and acc_order and hasattr(w_pk, "block") and ln is not None and aligned16(*ln)
    if (short and N <= attention_block_tokens(dt, H, head_dim, C, c_out)
            and resid is not None and resid.data_ptr() == x.data_ptr() and o_map is None
            and a_so % 16 == 0 and a_si % 16 == 0 and (C == 256 or bias_t is not None or bias_in_launch)
            and not (bias_in_launch and C == 256)          # ffk_pair_bias, which makes that bias, is built for 64 and 128 channels
            and (drop is None or drop.shape[0] == N)):
        if bias_in_launch:
            bias_t = alloc((H, NT, NT, 1024), dt, dev)
            _pair_bias_launch(bias_t, x, ln, w_pk[4 * ((H * 32 + 127) // 128) * 128:], pb_scratch, N=N, C=C, H=H, a_inner=a_inner,
                              a_so=a_so, a_si=a_si, scale=LOG2E)
        kb, flags = key_bias(mask, dev, B2=B2, N=N, mask_sb=mask_sb, mask_sn=mask_sn)
        w, bg = w_pk.block
        _lib.attention_block(out, x, ln[0], ln[1], w, bg, out_bias_pk, bias_t, kb, flags, B2=B2, N=N, C=C, D=head_dim,
                             s_row=a_so if a_inner == N else N * a_si, s_tok=a_si, bias_pitch=NT, xtail=xtail, drop=drop)
        return out
    qk_kind = FFK_TILE_ACC if acc_order else FFK_TILE_QK
    # Packed heads: nothing is written or read for padding (extra-MSA stack, 8 heads of 8 channels: a quarter of the operand
    # bytes; template stack, 4 heads of 16: half of them).
    packed = acc_order and hasattr(w_pk, "packed_heads")
    if packed:
        w_pk, gate_bias_pk, wo_pk = w_pk.packed_heads
    HC = H * head_dim if packed else H * 32
    if HC % 128 != 0 and not packed:
        raise RuntimeError("attention: n_head * 32 must be a multiple of 128 (got %d heads)" % H)
    # Rows of 256 channels too long for that, with a pair bias: one kernel up to the gated heads, the output projection behind it.
    heads = (short and C == 256 and head_dim == 32 and HC == C and N <= ATTENTION_HEADS_TOKENS and bias_t is not None
             and not bias_in_launch)
    HT = HC // 32                                  # operand tiles per batch row and 32 tokens
    per_row = 5 * HT * NT * 1024 * es
    slab = B2 if budget is None else min(B2, max(2, (budget // per_row) // 2 * 2))
    q_t, k_t, v_t = (alloc((slab, HT, NT, 1024), dt, dev, zero) for _ in range(3)) if not heads else (None,) * 3
    # Where the update goes back into the tensor the gate is computed from (every attention of the Evoformer block),
    # the gate is not a tensor at all: the output stage computes sigmoid(Wg LN(x) + bg) from the rows of x it reads as
    # residual anyway and multiplies the heads' outputs by it on their way into the output projection
    # (ffk_gated_out_fused).  The projection launch then writes q, k, v only and the core reads no gate.
    # Measured at N_seq = 128, same box: on the triangle attentions at N_res = 1024 the projection and the core each get
    # ~ 3 % faster and the output stage as much slower - 1.1 GB less memory traffic per block at the same block time; at
    # N_res = 256 a block gains 1.4 % (0.631 vs 0.640 ms) since the output stage runs three workgroups per CU (with two
    # it lost 1.3 %); on the MSA attentions (256 channels, two workgroups per CU) it loses slightly at both sizes.
    # Shorter rows were not measured and keep the gate tensor.  The choice depends on the row length and the width only, never on the number of
    # batch rows: a subset of the batch rows must give the bits of the full call.
    gate_in_out = (_GATE_IN_OUT_STAGE and drop is None and N >= _GATE_IN_OUT_MIN_N and C in _GATE_IN_OUT_WIDTHS and acc_order
                   and ln is not None and not packed and HC == C and c_out == C and resid is not None and o_map is None
                   and resid.data_ptr() == x.data_ptr() and a_so % 16 == 0 and a_si % 16 == 0 and not heads)
    gate = None
    if not gate_in_out and not heads:
        gate = alloc((slab, HT, NT, 1024) if acc_order else (slab * N, HC), dt, dev)
    o = alloc((slab * N, HC), dt, dev)
    tpg = (HC + 127) // 128
    qscale = LOG2E / math.sqrt(float(head_dim))
    tkw = dict(inner=N, s_o=HT * NT * 1024, s_h=NT * 1024, ncols=min(128, HC))
    bias_tile = None
    # rows of a bias buffer the caller leaves to this function (bias_in_launch with bias_t None) end in one unused tile
    # when the projection launch writes them: with 2^n key tiles per row every query-tile row would start in the same
    # memory channel (-2 % per triangle-attention launch at N = 1024, measured three times on one box)
    can_ride = (bias_in_launch and acc_order and C == 128 and H <= 4 and _PAIR_BIAS_RIDES
                and (not gate_in_out or hasattr(w_pk, "without_gate")))
    will_ride = can_ride and slab >= B2
    bias_padded = will_ride and _BIAS_ROW_PAD and bias_t is None
    if bias_in_launch:
        ntp = NT + (1 if bias_padded else 0)
        if bias_t is None:
            bias_t = alloc((H, NT, ntp, 1024), dt, dev, zero=(N % 32) != 0)
        bias_tile = make_tile(bias_t, kind=FFK_TILE_BIAS, inner=N, s_o=ntp * 1024, s_h=NT * ntp * 1024, ncols=H,
                              scale=LOG2E)
    # With 128 input channels, at most four heads and all rows in one slab the bias rides on the projection launch:
    # the weights-stationary kernel computes its four dot products per row (small MFMAs) from the rows it
    # has in LDS anyway (one read of x less than a pass of its own; -0.05 ms per triangle attention at N = 1024).
    rides = will_ride
    # Otherwise the skinny bias projection has its own pass over x.  It goes first: x was written by the launch before
    # this call and is still (partly) cache-resident, and the bias pass writes little, so the projection after
    # it finds x as warm as before - the other way round the projection's output (four times the size of x)
    # has pushed x out by the time the bias pass reads it (measured: -0.65 % block time at N = 1024).
    if rides:
        if pb_scratch is not None and not pb_scratch.ready:
            # The weight operand of the bias pass that short rows take, made with the other weights: made in the first pass of
            # another size it keeps that pass from being recorded.  The bias of one row, thrown away.
            _pair_bias_launch(alloc((H, 1, 1, 1024), dt, dev), x, ln, w_pk[4 * tpg * 128:], pb_scratch, N=1, C=C, H=H, a_inner=1,
                              a_so=0, a_si=C, scale=LOG2E)
    elif can_ride and N < 1024:
        # In slabs: the same kernel with the bias as its only tile, so that slabs change no bit of the result.  Longer rows
        # keep the bias pass of its own, which streams x twice as fast (16 M rows at N = 4096: 0.9 against 1.9 ms).
        _lib.fused_linear(x, w_pk, [bias_tile], M=M, K=C, a_inner=a_inner, a_so=a_so, a_si=a_si, ln=ln,
                          w_row_off=4 * tpg * 128)
        bias_tile = None
    elif bias_tile is not None and acc_order and C in (64, 128):
        _pair_bias_launch(bias_t, x, ln, w_pk[4 * tpg * 128:], pb_scratch, N=N, C=C, H=H, a_inner=a_inner,
                          a_so=a_so, a_si=a_si, scale=LOG2E)
        bias_tile = None
    if bias_tile is not None and not rides and (acc_order or slab < B2):     # its own launch over all rows, before x changes
        _lib.fused_linear(x, w_pk, [bias_tile], M=M, K=C, a_inner=a_inner, a_so=a_so, a_si=a_si, ln=ln,
                          w_row_off=4 * tpg * 128)
        bias_tile = None
    kb, flags = key_bias(mask, dev, B2=B2, N=N, mask_sb=mask_sb, mask_sn=mask_sn)
    for b0 in range(0, B2, slab):
        nb = min(slab, B2 - b0)
        Ms = nb * N
        # rows b0 * N ... of the map: a shifted base, and an inner extent that still covers the slab
        off, inner = (b0 * N * a_si, Ms) if a_inner == M else (b0 * a_so, N)
        o_off = b0 * N * o_si if a_inner == M else b0 * o_so
        if heads:
            w, bg = w_pk.block
            _lib.attention_heads(o, x.data_ptr() + off * es, ln[0], ln[1], w, bg, bias_t, kb[b0:b0 + nb], flags[b0:b0 + nb], B2=nb,
                                 N=N, C=C, D=head_dim, s_row=a_so if a_inner == N else N * a_si, s_tok=a_si, bias_pitch=NT)
        tiles = []
        for buf, kind, scale in () if heads else ((q_t, qk_kind, qscale), (k_t, qk_kind, 1.0), (v_t, FFK_TILE_V, 1.0)):
            for t in range(tpg):
                tiles.append(make_tile(buf.data_ptr() + t * 4 * NT * 1024 * es, kind=kind, scale=scale, **tkw))
        for t in range(0 if gate_in_out or heads else tpg):
            if acc_order:
                tiles.append(make_tile(gate.data_ptr() + t * 4 * NT * 1024 * es, kind=FFK_TILE_ACC,
                                       bias=gate_bias_pk.data_ptr() + t * 128 * es, act=FFK_ACT_SIGMOID, **tkw))
            else:
                tiles.append(make_tile(gate.data_ptr() + t * 128 * es, bias=gate_bias_pk.data_ptr() + t * 128 * es,
                                       inner=Ms, s_i=HC, act=FFK_ACT_SIGMOID))
        if bias_tile is not None:      # single slab: the bias rides on the projection launch
            tiles.append(bias_tile)
        per = _lib.WS_TILES if (acc_order and C == 256) else len(tiles)
        for t0 in range(0, len(tiles), per):
            # a bias tile riding behind q, k, v (no gate tiles) takes its weight rows from the gate-less packing
            wp = w_pk.without_gate if (gate_in_out and bias_tile is not None) else w_pk
            _lib.fused_linear(x, wp, tiles[t0:t0 + per], M=Ms, K=C, a_inner=inner, a_so=a_so, a_si=a_si, ln=ln,
                              w_row_off=t0 * 128, a_off=off)
        if not heads:
            _lib.attention_fwd(o, q_t, k_t, v_t, bias_t, kb[b0:b0 + nb], flags[b0:b0 + nb], gate, B2=nb, H=H, Nq=N, Nk=N,
                               gate_tiled=acc_order, bias_padded=bias_padded,
                               D=head_dim if packed else 32, half_k=not packed and head_dim <= (16 if acc_order else 8))
        if gate_in_out:
            # packed rows of w_pk: q, k, v, gate blocks of HC rows each; o holds the slab's rows in logical order
            _lib.gated_out_fused(out.data_ptr() + o_off * es, x.data_ptr() + off * es, ln[0], ln[1],
                                 w_pk.data_ptr() + 3 * HC * C * es, gate_bias_pk, o, wo_pk, out_bias_pk, M=Ms, C=C,
                                 inner=inner, s_o=a_so, s_i=a_si,
                                 xtail=None if xtail is None else xtail.data_ptr() + o_off)
            continue
        tiles = []
        for t in range((c_out + 127) // 128):
            tiles.append(make_tile(out.data_ptr() + (o_off + t * 128) * es,
                                   bias=None if out_bias_pk is None else out_bias_pk.data_ptr() + t * 128 * es,
                                   resid=None if resid is None else resid.data_ptr() + (o_off + t * 128) * es,
                                   xtail=xtail_ptr(xtail, o_off + t * 128),
                                   gate=None if drop is None else drop.data_ptr() + t * 128 * es,
                                   gate_ld=0 if drop is None else c_out, gate_rows=0 if drop is None else drop.shape[0],
                                   inner=inner, s_o=o_so, s_i=o_si, ncols=min(128, c_out - t * 128)))
        _lib.fused_linear(o, wo_pk, tiles, M=Ms, K=HC)
    return out


def pair_bias(z, *, r, C, H, ln, wb_pk, pb_scratch=None):
    """bias_t[h][q/32][k/32][tile] = log2e * (LN(z)[q, k, :] . Wb[h, :]) in score-accumulator tiles."""
    NT = (r + 31) // 32
    bias_t = alloc((H, NT, NT, 1024), z.dtype, z.device, zero=(r % 32) != 0)
    if z.dtype == torch.bfloat16 and C in (64, 128) and H <= 8:
        _pair_bias_launch(bias_t, z, ln, wb_pk, pb_scratch, N=r, C=C, H=H, a_inner=r * r, a_so=0, a_si=C, scale=LOG2E)
        return bias_t
    tile = make_tile(bias_t, kind=FFK_TILE_BIAS, inner=r, s_o=NT * 1024, s_h=NT * NT * 1024, ncols=H, scale=LOG2E)
    _lib.fused_linear(z, wb_pk, [tile], M=r * r, K=C, ln=ln)
    return bias_t


# ----------------------------------------------------------- triangle multiplication ----
def pack_trimul(proj_w, proj_b, gate_w, gate_b, og_w, og_b, c, dtype, device):
    """[left GLU tiles | right GLU tiles | output-gate tiles]; a GLU tile packs 64 channels as
    [p c0..c0+31 | g c0..c0+31 | p c0+32..c0+63 | g c0+32..c0+63]."""
    if c % 64 != 0:
        raise RuntimeError("triangle multiplication: hidden width must be a multiple of 64, got %d" % c)
    ws, bs = [], []
    for side in range(2):
        for t in range(c // 64):
            for q in range(2):
                sl = slice(side * c + t * 64 + q * 32, side * c + t * 64 + q * 32 + 32)
                ws += [proj_w[sl], gate_w[sl]]
                bs += [proj_b[sl], gate_b[sl]]
    n_glu = 2 * (c // 64)
    w = pack_rows(ws, dtype, device)
    b = pack_vec(bs, dtype, device)
    wg = pack_rows([og_w], dtype, device)
    bg = pack_vec([og_b], dtype, device)
    return torch.cat([w, wg], 0).contiguous(), torch.cat([b, bg], 0).contiguous(), n_glu


def pack_trimul_out(out_w, out_b, og_w, og_b, C, dtype, device, ln_p, ln_z):
    """Output stage with the gate computed in the same launch: GLU tiles of 64 channels,
    [Wout c0..c0+31 | Wog c0..c0+31 | Wout c0+32..c0+63 | Wog c0+32..c0+63] (biases alike), with both
    LayerNorms folded in: ``ln_p = (gamma, beta)`` of the contraction result into the value rows, ``ln_z`` of the
    pair tensor into the gate rows (W' = W * gamma rounded to the kernel dtype, b' = W beta + b).  Returns
    (weights, biases, fp32 row sums of W' in the same packed order)."""
    def fold(w, b, ln):
        w, b = w.detach().float(), b.detach().float()
        gam, bet = ln[0].detach().float(), ln[1].detach().float()
        wf = (w * gam[None, :]).to(dtype).float()
        return wf, w @ bet + b, wf.sum(1)
    out_w, out_b, out_rs = fold(out_w, out_b, ln_p)
    og_w, og_b, og_rs = fold(og_w, og_b, ln_z)
    ws, bs, cs = [], [], []
    for t in range(C // 64):
        for q in range(2):
            sl = slice(t * 64 + q * 32, t * 64 + q * 32 + 32)
            ws += [out_w[sl], og_w[sl]]
            bs += [out_b[sl], og_b[sl]]
            cs += [out_rs[sl], og_rs[sl]]
    return pack_rows(ws, dtype, device), pack_vec(bs, dtype, device), pack_vec(cs, torch.float32, device)


def trimul_gate_in_output_stage(dtype, r, C, c):
    """The output gate sigmoid(Wg LN(z) + bg) can be computed inside the output stage (second operand
    of the projection kernel) instead of being written by the first stage and read back."""
    return dtype == torch.bfloat16 and C == 128 and c == 128 and r % 8 == 0


# Elements between the channel planes of the triangle multiplication's operands and of its contraction result, beyond the
# r * kpad the data needs.  With planes exactly 2 MB apart (N_res = 1024, bf16) the 32 lanes of a channel-major store of
# the projection kernel - one channel each - all land in the same memory channel; 128 bytes of padding spread them
# (block 6.97 -> 6.885 ms in a same-box A/B at N_res = 1024; 64, 192 and 1088 elements measure the same).
_TRIMUL_CHAN_PAD = 64
_PAIR_BIAS_RIDES = True      # see attention(): switch for same-box comparisons
_BIAS_ROW_PAD = True         # see attention(): switch for same-box comparisons
_GATE_IN_OUT_STAGE = True    # see attention(): False keeps the gate a tensor (written by the projection, read by the core)
_GATE_IN_OUT_MIN_N = 256         # shortest attended axis for which the gate moves into the output stage
_GATE_IN_OUT_WIDTHS = (128,)     # ... and the channel widths (the kernel is built for 128 and 256)


def triangle_multiplication(z, out, *, r, C, c, incoming, ln1, w_pk, b_pk, n_glu, ln2, wout_pk, out_bias_pk, mask,
                            dual_pk=None, xtail=None, drop=None):
    """out = z + sigmoid(Wg LN(z) + bg) * (Wout LN2(p) + b_out),  p[i,j,:] = sum_k a[i,k,:] b[j,k,:]
    (outgoing) or sum_k a[k,i,:] b[k,j,:] (incoming), a/b the masked gated projections.
    ``dual_pk`` = (weights, biases) of pack_trimul_out: the gate is then computed in the output stage.
    ``drop``: None, or [r, C] dropout multipliers shared by all rows i (the update of (i, j) is scaled by drop[j]): the
    gate tensor is multiplied by it, so the output stage is the one with a gate tensor."""
    dt, dev = z.dtype, z.device
    es = es_of(dt)
    M = r * r
    kpad = round_up(r, vec_of(dt))
    zero = kpad != r
    # channel planes of the operands and of the contraction result are cs elements apart (_TRIMUL_CHAN_PAD beyond r * kpad)
    cs = r * kpad + _TRIMUL_CHAN_PAD
    lr = alloc((2, c, cs), dt, dev, zero)
    dual = dual_pk is not None and drop is None and trimul_gate_in_output_stage(dt, r, C, c)
    g = None if dual else alloc((M, C), dt, dev)
    tiles = []
    if incoming:      # logical row (a, b) reads z[b, a]
        a_map, m_so, m_si = (r, C, r * C), 1, r
    else:
        a_map, m_so, m_si = (M, 0, C), r, 1
    for side in range(2):
        for t in range(c // 64):
            ti = side * (c // 64) + t
            tiles.append(make_tile(lr.data_ptr() + (side * c + t * 64) * cs * es,
                                   bias=b_pk.data_ptr() + ti * 128 * es, glu=1, ncols=64, inner=r, s_o=kpad, s_i=1,
                                   s_h=32 * cs, s_d=cs, rowmask=mask, m_so=m_so, m_si=m_si))
    gates = []
    for t in range((C + 127) // 128 if not dual else 0):
        kw = dict(inner=r, s_o=C, s_i=r * C) if incoming and drop is None else dict(inner=M, s_i=C)
        gates.append(make_tile(g.data_ptr() + t * 128 * es, bias=b_pk.data_ptr() + (n_glu + t) * 128 * es,
                               act=FFK_ACT_SIGMOID, ncols=min(128, C - t * 128),
                               gate=None if drop is None else drop.data_ptr() + t * 128 * es,
                               gate_ld=0 if drop is None else C, gate_rows=0 if drop is None else r, **kw))
    # With dropout the gate has to be a tensor (its rows times the multipliers) and gets a launch of its own, which reads and
    # normalises z once more.  Against the gate on the first launch and a scaling pass over it, the whole multiplication at
    # N_res = 256 / 512 / 1 024: 91 / 311 / 1 193 us here, 86 / 315 / 1 265 there (66 / 213 / 840 without dropout, where the gate
    # is computed in the output stage); the training forward of a block 675 / 1 915 / 7 370 us here, 670 / 1 968 / 7 550 there.
    if drop is None:
        tiles, gates = tiles + gates, []
    _lib.fused_linear(z, w_pk, tiles, M=M, K=C, a_inner=a_map[0], a_so=a_map[1], a_si=a_map[2], ln=ln1)
    if gates:      # with dropout multipliers of row m % r: the gate's rows in the order of z, whatever the first launch's is
        _lib.fused_linear(z, w_pk, gates, M=M, K=C, ln=ln1, w_row_off=n_glu * 128)
    p = alloc((c, cs), dt, dev)
    _lib.bgemm_nt(lr[0], lr[1], p, M=r, N=r, K=kpad, lda=kpad, ldb=kpad, batch=c, a_bs=cs, b_bs=cs,
                  o_bs=cs, s_i=kpad)
    del lr
    if dual:
        wd, bd, rowsums = dual_pk
        tiles = [make_tile(out.data_ptr() + t * 64 * es, bias=bd.data_ptr() + t * 128 * es, glu=1, ncols=64,
                           resid=z.data_ptr() + t * 64 * es, xtail=xtail_ptr(xtail, t * 64), inner=M, s_i=C)
                 for t in range(C // 64)]
        # both LayerNorms (of p and of z) are folded into the packed weights: no normalisation pass over either
        _lib.fused_linear(p, wd, tiles, M=M, K=c, a_inner=r, a_so=kpad, a_si=1, a_chanmajor=True, a_cs=cs,
                          ln_rowsums=rowsums, a2=z, a2_inner=M, a2_si=C)
        return out
    tiles = []
    for t in range((C + 127) // 128):
        tiles.append(make_tile(out.data_ptr() + t * 128 * es, bias=out_bias_pk.data_ptr() + t * 128 * es,
                               gate=g.data_ptr() + t * 128 * es, gate_ld=C, resid=z.data_ptr() + t * 128 * es,
                               xtail=xtail_ptr(xtail, t * 128), inner=M, s_i=C, ncols=min(128, C - t * 128)))
    _lib.fused_linear(p, wout_pk, tiles, M=M, K=c, a_inner=r, a_so=kpad, a_si=1, a_chanmajor=True, a_cs=cs,
                      ln=ln2)
    return out


# ------------------------------------------------------------------ outer product mean ----
def opm_normaliser(mask):
    """fp32 [r, r]: sum over the sequences of mask[s, i] mask[s, j]; once per ``mask_cache``."""
    s, r = mask.shape

    def build():
        spad = round_up(s, vec_of(mask.dtype))
        mt = torch.zeros(r, spad, dtype=mask.dtype, device=mask.device)
        mt[:, :s] = mask.t()
        nrm = torch.empty(r, r, dtype=torch.float32, device=mask.device)
        _lib.bgemm_nt(mt, mt, nrm, M=r, N=r, K=spad, lda=spad, ldb=spad, out_f32=True)
        return nrm
    return _mask_derived(mask, ("opm_norm", s, r), build)


def outer_product_mean(m, mask, z, out, *, s, r, C, Cz, ln, wab_pk, bab_pk, wo, bo, budget, eps=1e-3, wo_ed=None,
                       xtail=None):
    """out = z + (Wo vec(sum_s a[s,i,:] (x) b[s,j,:]) + bo) / (sum_s mask[s,i] mask[s,j] + eps),
    a, b the masked 32-channel projections of LN(m).  m is [s, r, C] rows, mask [s, r]."""
    dt, dev = m.dtype, m.device
    es = es_of(dt)
    spad = round_up(s, vec_of(dt))
    fused = wo_ed is not None and dt == torch.bfloat16 and Cz == 128 and r % 32 == 0 and s <= 128
    if fused:       # the fused kernel's sequence extents; the zero sequences add nothing to a sum
        spad = 64 if s <= 64 else 128
    ab = alloc((2, r * 32, spad), dt, dev, zero=spad != s)
    tile = make_tile(ab, bias=bab_pk, ncols=64, inner=s, s_o=32 * spad, s_i=1, s_h=r * 32 * spad, s_d=spad,
                     rowmask=mask, m_so=1, m_si=r)
    # logical row (i, s') reads m[s', i]
    _lib.fused_linear(m, wab_pk, [tile], M=s * r, K=C, a_inner=s, a_so=C, a_si=r * C, ln=ln)
    nrm = opm_normaliser(mask)
    if fused:
        # fused core: the [r, r, 1024] outer product never leaves the chip
        _lib.opm_fused(out, z, ab[0], ab[1], wo_ed, bo, nrm, r=r, spad=spad, eps=eps, xtail=xtail)
        return out
    ci = max(1, min(r, budget // (r * 1024 * es)))
    O = alloc((ci * r, 1024), dt, dev)
    for i0 in range(0, r, ci):
        n = min(ci, r - i0)
        _lib.bgemm_nt(ab.data_ptr() + i0 * 32 * spad * es, ab[1], O, M=32 * n, N=32 * r, K=spad, lda=spad, ldb=spad,
                      inner=32, s_o=r * 1024, s_i=32, s_h=1024, s_d=1, dtype=dt)
        _lib.bgemm_nt(O, wo, out.data_ptr() + i0 * r * Cz * es, M=n * r, N=Cz, K=1024, lda=1024, ldb=1024, bias=bo,
                      rowdiv=nrm.data_ptr() + i0 * r * 4, div_eps=eps, resid=z.data_ptr() + i0 * r * Cz * es, dtype=dt,
                      xtail=xtail_ptr(xtail, i0 * r * Cz))
    return out


# --------------------------------------------------------------- global attention ----
def global_attention(x, out, resid, *, S, R, C, H, D, x_ss, x_sr, out_ss, out_sr, ln, wq, wk, wv, wg_pk, gb_pk,
                     wo_pk, ob_pk, c_out, mask, mask_ss, mask_sr, eps, budget):
    """Global column attention (one mean query per column j, shared key / value head):
    out[s, j] = (resid[s, j] +) Wo (sigmoid(Wg LN(x[s, j]) + bg) * o[j]) + bo, o from
    ``ffk_global_attention_core``.  Row (s, j) of x is at ``s * x_ss + j * x_sr`` (elements), of out /
    resid at ``s * out_ss + j * out_sr``; ``ln = None`` takes x as already normalised."""
    dt, dev = x.dtype, x.device
    es = es_of(dt)
    HD = H * D
    if not fits_fused(C, dt) or not fits_fused(HD, dt) or HD > 128 or c_out % vec_of(dt) != 0:
        raise RuntimeError("global_attention: unsupported widths C=%d, H*D=%d, out=%d" % (C, HD, c_out))
    o = alloc((R, HD), dt, dev)
    _lib.global_attention_core(o, x, mask, None if ln is None else ln[0], None if ln is None else ln[1], wq, wk, wv,
                               S=S, R=R, C=C, H=H, D=D, m_ss=x_ss, m_sr=x_sr, mask_ss=mask_ss, mask_sr=mask_sr,
                               scaling=D ** -0.5, eps=eps)
    # gate and output projection, a bounded number of sequences at a time
    sc = max(1, min(S, budget // max(1, R * HD * es)))
    tmp = alloc((sc * R, HD), dt, dev)
    for s0 in range(0, S, sc):
        n = min(sc, S - s0)
        M = n * R
        gate_tile = make_tile(tmp, bias=gb_pk, inner=M, s_i=HD, act=FFK_ACT_SIGMOID, ncols=HD, gate=o, gate_ld=HD,
                              gate_rows=R)
        _lib.fused_linear(x, wg_pk, [gate_tile], M=M, K=C, a_inner=R, a_so=x_ss, a_si=x_sr, ln=ln, a_off=s0 * x_ss)
        tiles = []
        for t in range((c_out + 127) // 128):
            tiles.append(make_tile(out.data_ptr() + (s0 * out_ss + t * 128) * es,
                                   bias=None if ob_pk is None else ob_pk.data_ptr() + t * 128 * es,
                                   resid=None if resid is None else resid.data_ptr() + (s0 * out_ss + t * 128) * es,
                                   inner=R, s_o=out_ss, s_i=out_sr, ncols=min(128, c_out - t * 128)))
        _lib.fused_linear(tmp, wo_pk, tiles, M=M, K=HD)
    return out
