"""Evoformer block and 48-block stack with the reference's interface
(fastfold/model/fastnn/evoformer.py:17-332), single GPU (DAP size 1).

Padding contract.  The reference pads the residue axis by ``padding_size = 1`` in the first
block even at DAP size 1, carries ``[1, s, r+1, c]`` / ``[1, r+1, r+1, c]`` tensors between
blocks and strips the pad in the last block (evoformer.py:42-62,78-89).  The padded key is
masked in every attention and every masked projection, and padded rows are discarded, so
results on the un-padded region do not depend on it.  ``Evoformer.forward`` keeps that
*interface* (same shapes in and out for first / middle / last blocks) but computes on the
un-padded region only; ``EvoformerStack`` never materialises the pad at all.
"""
from typing import Optional, Tuple

import torch
import torch.nn as nn
import torch.nn.functional as F
from torch.utils.checkpoint import checkpoint

from fastfold_amd import _plan
from . import _backward
from . import _fused as F_
from .msa import MSACore
from .ops import Linear, OutProductMean, _budget, _mask_like, _needs_grad, _no_grad_guard
from .triangle import PairCore


def _private_copy(view, owner):
    out = view.contiguous()
    return out.clone() if out.data_ptr() == owner.data_ptr() else out


def _save(ctx, block, keys, m, z, msa_mask, pair_mask, multipliers):
    """Keeps what the backward pass of a block reads; the multipliers as the dict ``drops`` (None without ``keys``).  All of it
    through ``save_for_backward``: a mask that is changed in place between the passes is an error, not another gradient."""
    ctx.block, ctx.keys = block, keys
    ctx.save_for_backward(m, z, msa_mask, pair_mask, *multipliers)
    return None if keys is None else dict(zip(keys, multipliers))


def _saved(ctx):
    m, z, msa_mask, pair_mask, *multipliers = ctx.saved_tensors
    return m, z, (msa_mask, pair_mask), None if ctx.keys is None else dict(zip(ctx.keys, multipliers))


class _BlockRecompute(torch.autograd.Function):
    """One Evoformer block as its own checkpoint, for blocks ``_backward.block_backward`` does not cover: the forward pass runs
    the fused launches (nothing of it is kept but the two inputs, the masks and the dropout multipliers, which the caller draws
    so that both passes see the same ones); the backward pass re-runs the block module by module with autograd on, the way
    block checkpointing re-runs it (fastfold/utils/checkpointing.py:55-73; evoformer.py:262-266), and back-propagates through
    that."""

    @staticmethod
    def forward(ctx, block, keys, _grad_anchor, m, z, msa_mask, pair_mask, *multipliers):
        drops = _save(ctx, block, keys, m, z, msa_mask, pair_mask, multipliers)
        return block._core_any(m.contiguous(), z.contiguous(), msa_mask, pair_mask, inplace=False, drops=drops)

    @staticmethod
    def backward(ctx, dm, dz):
        m, z, masks, drops = _saved(ctx)
        with torch.enable_grad():
            m_, z_ = m.detach().requires_grad_(True), z.detach().requires_grad_(True)
            mo, zo = ctx.block._core_train(m_, z_, *masks, drops=drops if drops is not None else {})
        torch.autograd.backward((mo, zo), (dm, dz))        # parameter gradients accumulate here, as under checkpointing
        return (None, None, None, m_.grad, z_.grad, None, None, *(None for _ in ctx.keys or ()))


class _BlockGrad(torch.autograd.Function):
    """One Evoformer block as its own checkpoint, forward and backward as launch sequences (``_backward.block_backward``): the
    forward pass keeps the two inputs, the masks and the dropout multipliers (drawn by the caller), the backward pass returns the
    gradients of the inputs and of every parameter."""

    @staticmethod
    def forward(ctx, block, keys, m, z, msa_mask, pair_mask, *rest):
        n = len(keys or ())
        ctx.params = rest[n:]
        drops = _save(ctx, block, keys, m, z, msa_mask, pair_mask, rest[:n])
        return block._core_any(m.contiguous(), z.contiguous(), msa_mask, pair_mask, inplace=False, drops=drops)

    @staticmethod
    def backward(ctx, dm, dz):
        m, z, masks, drops = _saved(ctx)
        dm, dz, grads = ctx.block._backward(m, z, *masks, dm, dz, drops)
        need = ctx.needs_input_grad
        first = 6 + len(ctx.keys or ())
        grads = [g.to(p.dtype) if need[first + i] else None for i, (p, g) in enumerate(zip(ctx.params, grads))]
        return (None, None, dm if need[2] else None, dz if need[3] else None, None, None, *(None for _ in ctx.keys or ()), *grads)


class Evoformer(nn.Module):

    # A call that autograd has to see is its own checkpoint: it runs the fused forward and keeps the block's inputs
    # (_BlockGrad, _BlockRecompute).  False: the forward is the chain of the block's modules, each of which keeps its own
    # input, and the backward pass does not re-run the block.
    recompute_in_backward = True

    def __init__(self, c_m: int, c_z: int, first_block: bool, last_block: bool, is_multimer: bool = False):
        super(Evoformer, self).__init__()
        self.first_block = first_block
        self.last_block = last_block
        self.msa = MSACore(c_m, c_z, p_drop=0.15)
        self.communication = OutProductMean(n_feat=c_m, n_feat_out=c_z, n_feat_proj=32)
        self.pair = PairCore(d_pair=c_z)
        self.is_multimer = is_multimer

    # -- un-padded core on [1, s, r, c_m] / [1, r, r, c_z] / [1, s, r] / [1, r, r] ----------
    def _core(self, m, z, msa_mask, pair_mask, inplace: bool, tails=(None, None), drops=None):
        """``tails = (m_tail, z_tail)``: int8 tails of m / z as extended residual streams (the stack's bf16 mode),
        or None for the plain stream of the reference.  ``drops``: None, or the dropout multipliers of a training-mode
        pass (``_draw_drops``)."""
        F_.check_nonempty("Evoformer", m, z)
        F_.check_cuda(m, z, msa_mask, pair_mask)
        _no_grad_guard(self, m, z)
        m_out, z_out = (m, z) if inplace else (torch.empty_like(m), torch.empty_like(z))
        s, r = m.shape[1], m.shape[2]
        msa_mask, pair_mask = _mask_like(msa_mask, m), _mask_like(pair_mask, z)
        with F_.mask_scope():
            mm, pm = msa_mask[0], pair_mask[0]
            drop = [(drops or {}).get(k) for k in ("row", "tmo", "tmi", "tas", "tae")]
            tensors = [m, z, m_out, z_out, *tails, mm, pm, *F_.key_bias(mm, m.device, B2=s, N=r, mask_sb=r, mask_sn=1),
                       *F_.key_bias(mm, m.device, B2=r, N=s, mask_sb=1, mask_sn=r),
                       *F_.key_bias(pm, m.device, B2=r, N=r, mask_sb=r, mask_sn=1),
                       *F_.key_bias(pm, m.device, B2=r, N=r, mask_sb=1, mask_sn=r), F_.opm_normaliser(mm), *drop]
            key = (m.shape, z.shape, mm.shape, pm.shape, m.dtype, m.device, inplace, self.is_multimer, _budget(), F_.switches(),
                   tuple(t is None for t in (*tails, *drop)))
            _plan.run(self, key, tensors, lambda: self._sequence(m, z, m_out, z_out, msa_mask, pair_mask, tails, drops))
        return m_out, z_out

    def _sequence(self, m, z, m_out, z_out, msa_mask, pair_mask, tails, drops):
        mt, zt = tails
        if self.is_multimer:
            # multimer order (evoformer.py:70-76, 133-137): outer product mean first, the MSA stack reads the
            # pair tensor it leaves, the pair stack runs last
            self.communication._run(m, msa_mask, z, z_out, zt)
            self.msa._into(m, z_out, msa_mask, m_out, mt, drops)
        else:
            self.msa._into(m, z, msa_mask, m_out, mt, drops)
            self.communication._run(m_out, msa_mask, z, z_out, zt)
        self.pair.inplace([z_out], pair_mask, zt, drops=drops)

    def _core_any(self, m, z, msa_mask, pair_mask, inplace: bool, drops=None):
        """``_core`` at any extents: ragged bf16 tensors run zero-padded to whole tiles (``_fused.pad_to_tiles``)."""
        s, r = m.shape[1], m.shape[2]
        mp, zp, mk, pk = F_.pad_to_tiles(m, z, msa_mask, pair_mask)
        if mp is m and zp is z:
            return self._core(m, z, msa_mask, pair_mask, inplace, drops=drops)
        if drops and zp is not z:
            # multipliers of the padding rows: any will do
            drops = {k: F.pad(v, (0, 0, 0, zp.shape[1] - r) if v.shape[1] == 1 else (0, 0, 0, 0, 0, zp.shape[1] - r))
                     for k, v in drops.items()}
        mp, zp = self._core(mp, zp, mk, pk, inplace=inplace or (mp is not m and zp is not z), drops=drops)
        mp, zp = mp[:, :s, :r], zp[:, :r, :r]
        if inplace:
            return m.copy_(mp) if mp.data_ptr() != m.data_ptr() else m, z.copy_(zp) if zp.data_ptr() != z.data_ptr() else z
        return mp.contiguous(), zp.contiguous()

    def _core_train(self, m, z, msa_mask, pair_mask, drops=None):
        """The differentiable block (evoformer.py:64-76) on the un-padded tensors: every update is out of place and
        made of operators with a backward pass.  ``drops``: None (every module draws its own dropout mask in training
        mode) or the multipliers drawn by the caller (a dict, possibly empty: no dropout)."""
        F_.check_nonempty("Evoformer", m, z)
        if self.is_multimer:
            z_ori = self.communication(m, msa_mask, z)
            z = self.pair(z_ori, pair_mask, drops=drops)
            return self.msa(m, z_ori, msa_mask, drops=drops), z
        m = self.msa(m, z, msa_mask, drops=drops)
        z = self.communication(m, msa_mask, z)
        return m, self.pair(z, pair_mask, drops=drops)

    def _backward(self, m, z, msa_mask, pair_mask, dm, dz, drops):
        """Gradients of a pass of this block on the un-padded tensors: (dm, dz, [one per ``_backward.parameters``]).  Extents
        that are no multiples of 32 run zero-padded (a masked position has no gradient and gives none)."""
        s, r = m.shape[1], m.shape[2]
        ds, dr = F_.round_up(s, 32) - s, F_.round_up(r, 32) - r
        with torch.no_grad():
            m, z, dm, dz = m.contiguous(), z.contiguous(), dm.to(m.dtype).contiguous(), dz.to(z.dtype).contiguous()
            msa_mask, pair_mask = _mask_like(msa_mask, m), _mask_like(pair_mask, z)
            if ds or dr:
                m, dm = (F.pad(t, (0, 0, 0, dr, 0, ds)) for t in (m, dm))
                msa_mask = F.pad(msa_mask, (0, dr, 0, ds))
            if dr:
                z, dz = (F.pad(t, (0, 0, 0, dr, 0, dr)) for t in (z, dz))
                pair_mask = F.pad(pair_mask, (0, dr, 0, dr))
                drops = {k: F.pad(v, (0, 0, 0, dr) if v.shape[1] == 1 else (0, 0, 0, 0, 0, dr)) for k, v in (drops or {}).items()}
            dm_in, dz_in = torch.empty_like(m), torch.empty_like(z)
            st = self.__dict__.get("_grad_layout")
            params = _backward.parameters(self)
            if st is None or [id(p) for p in st.params] != [id(p) for p in params]:
                st = _backward.Grads(params)
                self.__dict__["_grad_layout"] = st
            g = st.bind(torch.empty(st.numel, dtype=m.dtype, device=m.device))
            sp, rp = m.shape[1], m.shape[2]
            with F_.mask_scope():
                mm, pm = msa_mask[0], pair_mask[0]
                derived = [F_.key_bias(mm, m.device, B2=sp, N=rp, mask_sb=rp, mask_sn=1),
                           F_.key_bias(mm, m.device, B2=rp, N=sp, mask_sb=1, mask_sn=rp),
                           F_.key_bias(pm, m.device, B2=rp, N=rp, mask_sb=rp, mask_sn=1),
                           F_.key_bias(pm, m.device, B2=rp, N=rp, mask_sb=1, mask_sn=rp), F_.opm_normaliser(mm)]
                drop = [(drops or {}).get(k) for k in ("row", "tmo", "tmi", "tas", "tae")]
                tensors = [m, z, dm, dz, dm_in, dz_in, g.flat, mm, pm, *(t for pair in derived[:4] for t in pair), derived[4], *drop]
                key = ("backward", m.shape, z.shape, mm.shape, pm.shape, m.dtype, m.device, self.is_multimer, _budget(),
                       F_.switches(), tuple(t is None for t in drop))
                _plan.run(self, key, tensors, lambda: _backward.block_backward(
                    self, m, z, msa_mask, pair_mask, dm, dz, dm_in, dz_in, g, drops, derived=derived, budget=_budget()))
            if ds or dr:
                dm_in = dm_in[:, :s, :r].contiguous()
            if dr:
                dz_in = dz_in[:, :r, :r].contiguous()
        return dm_in, dz_in, g.views()

    def _draw_drops(self, m, z):
        """Dropout multipliers (0 or 1 / (1 - p)) of one training-mode pass of this block, one tensor per update that
        the reference drops (msa.py:70-73; triangle.py:66-75,122-131,168-173,215-222): shared along the rows, except for
        the ending-node attention, which shares them along the columns.  None in eval mode."""
        if not self.training:
            return None
        r = z.shape[-2]

        def draw(p, shape):
            return F.dropout(torch.ones(shape, dtype=z.dtype, device=z.device), p=p, training=True) if p > 0 else None
        pair = self.pair
        d = {"row": draw(self.msa.MSARowAttentionWithPairBias.p_drop, (1, 1, r, m.shape[-1])),
             "tmo": draw(pair.TriangleMultiplicationOutgoing.p_drop, (1, 1, r, z.shape[-1])),
             "tmi": draw(pair.TriangleMultiplicationIncoming.p_drop, (1, 1, r, z.shape[-1])),
             "tas": draw(pair.TriangleAttentionStartingNode.p_drop, (1, 1, r, z.shape[-1])),
             "tae": draw(pair.TriangleAttentionEndingNode.p_drop, (1, r, 1, z.shape[-1]))}
        return {k: v for k, v in d.items() if v is not None}

    def _run_grad(self, m, z, msa_mask, pair_mask):
        """The block under autograd, on the un-padded [1, ...] tensors."""
        if not self.recompute_in_backward:
            return self._core_train(m, z, msa_mask, pair_mask)
        if not _backward.as_built(self):
            # hooks or exchanged modules somewhere in the block: the fused launches would pass them by
            return checkpoint(self._core_train, m, z, msa_mask, pair_mask, use_reentrant=False)
        msa_mask, pair_mask = _backward.kept(msa_mask, m), _backward.kept(pair_mask, z)
        drops = self._draw_drops(m, z)
        keys, multipliers = (None, ()) if drops is None else (tuple(drops), tuple(drops.values()))
        if m.dtype in (torch.bfloat16, torch.float32) and z.dtype == m.dtype and m.shape[-1] == 256 and z.shape[-1] == 128:
            params = _backward.parameters(self)
            if _backward.supported(self, params):
                return _BlockGrad.apply(self, keys, m, z, msa_mask, pair_mask, *multipliers, *params)
        anchor = torch.empty(0, device=m.device, requires_grad=True)     # outputs need a gradient even when m and z do not
        return _BlockRecompute.apply(self, keys, anchor, m, z, msa_mask, pair_mask, *multipliers)

    def _enter(self, m, z, r):
        if self.first_block:
            return m.unsqueeze(0).contiguous(), z.unsqueeze(0).contiguous()
        if m.dim() != 4 or z.dim() != 4 or m.shape[2] != r + 1 or z.shape[1] != r + 1:
            raise RuntimeError("Evoformer: a non-first block expects padded [1, s, r+1, c] / [1, r+1, r+1, c] "
                               "inputs, got %s / %s" % (tuple(m.shape), tuple(z.shape)))
        # the core runs in place on these: they must be copies even where the un-padding slice is already
        # contiguous (a single sequence, a single residue) and ``.contiguous()`` would hand back the caller's memory
        return _private_copy(m[:, :, :r, :], m), _private_copy(z[:, :r, :r, :], z)

    def _leave(self, m, z):
        if self.last_block:
            return m.squeeze(0), z.squeeze(0)
        return F.pad(m, (0, 0, 0, 1)), F.pad(z, (0, 0, 0, 1, 0, 1))

    def forward(self, m: torch.Tensor, z: torch.Tensor, msa_mask: torch.Tensor, pair_mask: torch.Tensor,
                chunk_size: Optional[int] = None, _mask_trans: bool = True) -> Tuple[torch.Tensor, torch.Tensor]:
        """``chunk_size`` and ``_mask_trans`` are accepted and ignored, as in the reference
        (evoformer.py:36-37): chunking is the process-global ``set_chunk_size`` and transitions
        are never masked."""
        r = pair_mask.size(-1)
        if _needs_grad(self, m, z):
            if self.first_block:
                m, z = m.unsqueeze(0), z.unsqueeze(0)
            else:
                m, z = m[:, :, :r, :], z[:, :r, :r, :]
            return self._leave(*self._run_grad(m, z, msa_mask.unsqueeze(0), pair_mask.unsqueeze(0)))
        m, z = self._enter(m, z, r)
        m, z = self._core_any(m, z, msa_mask.unsqueeze(0), pair_mask.unsqueeze(0), inplace=not self.first_block)
        return self._leave(m, z)

    def inplace(self, m, z, msa_mask: torch.Tensor, pair_mask: torch.Tensor, chunk_size: Optional[int] = None,
                _mask_trans: bool = True):
        """List-passing variant (evoformer.py:93-152): ``m`` and ``z`` are one-element lists whose
        tensors are updated / rebound.  Memory beside them as for ``EvoformerStack.inplace``."""
        r = pair_mask.size(-1)
        if self.first_block:
            mm, zz = m[0].unsqueeze(0), z[0].unsqueeze(0)
            if not mm.is_contiguous() or not zz.is_contiguous():
                mm, zz = mm.contiguous(), zz.contiguous()
        else:
            mm, zz = self._enter(m[0], z[0], r)
        mm, zz = self._core_any(mm, zz, msa_mask.unsqueeze(0), pair_mask.unsqueeze(0), inplace=True)
        m[0], z[0] = self._leave(mm, zz)
        return m, z


class EvoformerStack(nn.Module):
    """Main Evoformer trunk (Algorithm 6): ``no_blocks`` blocks, then ``s = Linear(c_m, c_s)(m[0])``."""

    # bf16 / fp16 runs keep eight extra mantissa bits of both residual streams in int8 side tensors between the
    # blocks (see "extended residual stream" in include/ffk.h): rounding m and z to bf16 after each of the ~430
    # sub-updates of 48 blocks alone costs 2e-2 .. 3e-2 relative L2 at the output.  False = the reference's plain stream.
    extended_residual = True

    def __init__(self, c_m: int, c_z: int, c_s: int, no_blocks: int, blocks_per_ckpt: int,
                 clear_cache_between_blocks: bool = False, is_multimer: bool = False, **kwargs):
        super(EvoformerStack, self).__init__()
        self.blocks_per_ckpt = blocks_per_ckpt
        self.clear_cache_between_blocks = clear_cache_between_blocks
        self.blocks = nn.ModuleList()
        for block_id in range(no_blocks):
            self.blocks.append(Evoformer(c_m=c_m, c_z=c_z, first_block=(block_id == 0),
                                         last_block=(block_id == no_blocks - 1), is_multimer=is_multimer))
        self.linear = Linear(c_m, c_s)

    def _run(self, m, z, msa_mask, pair_mask, inplace_first: bool):
        F_.check_nonempty("EvoformerStack", m, z)
        s, r = m.shape[0], m.shape[1]
        m0, z0 = m.unsqueeze(0), z.unsqueeze(0)
        mm, zz, mk, pk = F_.pad_to_tiles(m0, z0, msa_mask.unsqueeze(0), pair_mask.unsqueeze(0))
        own_m, own_z = mm is not m0, zz is not z0        # padded copies may be overwritten
        tails = (None, None)
        if self.extended_residual and mm.dtype == torch.bfloat16 and mm.is_cuda:
            # zero tails: the inputs are exact bf16 values; the tails die with this call, the bf16 tensors they
            # leave are the correctly rounded results
            tails = (torch.zeros(mm.shape, dtype=torch.int8, device=mm.device),
                     torch.zeros(zz.shape, dtype=torch.int8, device=zz.device))
        with F_.mask_cache():          # key biases / normalisers depend on the masks only: once per stack, not per block
            for i, b in enumerate(self.blocks):
                if self.clear_cache_between_blocks:
                    torch.cuda.empty_cache()
                mm, zz = b._core(mm.contiguous(), zz.contiguous(), mk, pk, inplace=(inplace_first or i > 0 or (own_m and own_z)),
                                 tails=tails)
        mm, zz = mm.squeeze(0), zz.squeeze(0)
        if own_m:
            mm = m.copy_(mm[:s, :r]) if inplace_first else mm[:s, :r].contiguous()
        if own_z:
            zz = z.copy_(zz[:r, :r]) if inplace_first else zz[:r, :r].contiguous()
        return mm, zz

    def _run_train(self, m, z, msa_mask, pair_mask):
        """The differentiable stack: plain residual stream, blocks re-run in the backward pass in groups of
        ``blocks_per_ckpt`` while the module is in training mode (evoformer.py:262-266)."""
        mm, zz = m.unsqueeze(0), z.unsqueeze(0)
        mk, pk = msa_mask.unsqueeze(0), pair_mask.unsqueeze(0)
        blocks = list(self.blocks)
        per = self.blocks_per_ckpt if (self.training and self.blocks_per_ckpt) else None

        def run(group, a, b):
            for blk in group:
                if self.clear_cache_between_blocks:
                    torch.cuda.empty_cache()
                a, b = blk._core_train(a, b, mk, pk)
            return a, b
        if per is None:
            mm, zz = run(blocks, mm, zz)
        elif all(blk.recompute_in_backward for blk in blocks):
            # every block its own checkpoint, with a fused forward (at least as fine as groups of blocks_per_ckpt)
            for blk in blocks:
                if self.clear_cache_between_blocks:
                    torch.cuda.empty_cache()
                mm, zz = blk._run_grad(mm, zz, mk, pk)
        else:
            for i in range(0, len(blocks), per):
                mm, zz = checkpoint(run, blocks[i:i + per], mm, zz, use_reentrant=False)
        return mm.squeeze(0), zz.squeeze(0)

    def forward(self, m: torch.Tensor, z: torch.Tensor, msa_mask: torch.Tensor, pair_mask: torch.Tensor,
                chunk_size: int = None, _mask_trans: bool = True
                ) -> Tuple[torch.Tensor, torch.Tensor, Optional[torch.Tensor]]:
        """
        m [N_seq, N_res, C_m], z [N_res, N_res, C_z], msa_mask [N_seq, N_res], pair_mask [N_res, N_res]
        -> (m, z, s [N_res, C_s]).  Inputs are left untouched.
        """
        if _needs_grad(self, m, z):
            m, z = self._run_train(m, z, msa_mask, pair_mask)
            return m, z, self.linear(m[..., 0, :, :])
        m, z = self._run(m, z, msa_mask, pair_mask, inplace_first=False)
        s = self.linear(m[..., 0, :, :])
        return m, z, s

    def inplace(self, m, z, msa_mask: torch.Tensor, pair_mask: torch.Tensor, chunk_size: int = None,
                _mask_trans: bool = True):
        """``m`` / ``z`` are one-element lists; their tensors are overwritten (evoformer.py:280-332).  Beside them the call
        holds the scratch of one sub-module (at most about three pair tensors), in bf16 the tails of the residual streams (half
        the size of m and z) and, in bf16 at extents that are no multiples of 32, zero-padded copies of m and z: 15.3 GB at
        N_seq = 64, N_res = 4 096 and 19.8 GB at 4 090, where z has 4.3 GB."""
        contiguous = m[0].is_contiguous() and z[0].is_contiguous()
        mm, zz = self._run(m[0], z[0], msa_mask, pair_mask, inplace_first=contiguous)
        m[0], z[0] = mm, zz
        s = self.linear(m[0][..., 0, :, :])
        return m, z, s
