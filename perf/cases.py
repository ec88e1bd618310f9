"""Workloads of the Evoformer path as its users run it, for timing and for comparing outputs between versions.

A case is a dict of plain values; ``path`` names what is called:

  trunk      ``EvoformerStack`` inference: (m, z) -> (m, z, s), the trunk of one recycling iteration
  train      ``EvoformerStack`` in training mode: forward, backward, input and parameter gradients
  extra_msa  ``ExtraMSAStack`` inference: the 4-block stack over the unclustered sequences that feeds the trunk
  template   ``TemplatePairStack`` on up to four templates, then ``TemplatePointwiseAttention`` onto the pair tensor
  kernels    the stand-alone operators of ``fastnn.kernel`` (softmax, LayerNorm, attention core), forward and backward

Widths are the model's own (c_m = 256, c_z = 128, c_s = 384, c_e = 64, c_t = 64); weights ~ N(0, 0.02^2), LayerNorm
weights around one, inputs ~ N(0, 1), masks as a residue mask with a padded tail makes them.  A program loads its model
once and calls it with many inputs, so the modules are kept between preparations and only the inputs follow the seed.
"""
import math

import torch

from fastfold_amd.model.fastnn import (EvoformerStack, ExtraMSAStack, TemplatePairStack, TemplatePointwiseAttention,
                                       set_chunk_size)
from fastfold_amd.model.fastnn.kernel import LayerNorm, fused_attention_core, fused_softmax

C_M, C_Z, C_S, C_E, C_T = 256, 128, 384, 64, 64
DTYPES = {"bf16": torch.bfloat16, "fp32": torch.float32}
BYTES = {"bf16": 2, "fp32": 4}


def listed():
    return [
        # one block of a small domain in full precision: the reference configuration of the numerical checks, and the
        # smallest call (launch latency and host work count, not bandwidth)
        dict(name="block-fp32-r64", path="trunk", dtype="fp32", blocks=1, n_seq=32, n_res=64, tail=0.0, chunk=0),
        # the whole trunk on a short chain of odd length, as a scan over many small proteins calls it
        dict(name="trunk-bf16-r77", path="trunk", dtype="bf16", blocks=48, n_seq=128, n_res=77, tail=0.0, chunk=0),
        # the whole trunk at the crop size models are trained and benchmarked at
        dict(name="trunk-bf16-r256", path="trunk", dtype="bf16", blocks=48, n_seq=128, n_res=256, tail=0.0, chunk=0),
        # an ordinary chain at its own length (nothing rounds it), an odd number of sequences in its alignment;
        # the time per block does not depend on how many follow each other, so the larger cases run a part of the trunk
        dict(name="trunk-bf16-r391", path="trunk", dtype="bf16", blocks=8, n_seq=125, n_res=391, tail=0.0, chunk=0),
        # a long chain padded to a bucket length: the last residues are masked
        dict(name="trunk-bf16-r1024", path="trunk", dtype="bf16", blocks=4, n_seq=128, n_res=1024, tail=0.05, chunk=0),
        # a complex of several chains: bounded memory, so chunked and in place
        dict(name="trunk-bf16-r4096-inplace", path="trunk", dtype="bf16", blocks=1, n_seq=64, n_res=4096, tail=0.0, chunk=64),
        # full-precision inference at the crop size
        dict(name="trunk-fp32-r256", path="trunk", dtype="fp32", blocks=2, n_seq=128, n_res=256, tail=0.0, chunk=0),
        # a training step of stacked blocks at the crop size, dropout active
        dict(name="train-bf16-r256", path="train", dtype="bf16", blocks=4, n_seq=128, n_res=256, tail=0.0),
        # full-precision fine-tuning on a chain shorter than the crop, its tail masked
        dict(name="train-fp32-r117", path="train", dtype="fp32", blocks=2, n_seq=40, n_res=117, tail=0.1),
        # the extra-MSA stack of an ordinary chain with a deep alignment
        dict(name="extra-msa-bf16-r384", path="extra_msa", dtype="bf16", blocks=4, n_seq=1024, n_res=384, tail=0.0),
        # four templates of an ordinary chain, embedded and attended over by the pair tensor
        dict(name="template-bf16-r320", path="template", dtype="bf16", blocks=2, n_templ=4, n_res=320, tail=0.05),
        # the operators on their own at the size of the operator benchmark: 128 rows of 256 keys, 8 heads
        dict(name="kernels-bf16-n256", path="kernels", dtype="bf16", b2=128, heads=8, n=256),
    ]


def _spread(rng, lo, hi, whole_tiles):
    """An integer between lo and hi, spread over its logarithm; a multiple of 32 if ``whole_tiles``."""
    v = math.exp(rng.uniform(math.log(lo), math.log(hi)))
    return max(32, round(v / 32) * 32) if whole_tiles else round(v)


def draw(rng):
    path = rng.choice(["trunk", "trunk", "trunk", "train", "train", "extra_msa", "template", "kernels"])
    tiles = rng.random() < 0.3            # programs that crop or bucket; the others keep the chain's own length
    tail = rng.choice([0.0, 0.0, 0.05, 0.15])
    if path == "trunk":
        dtype = rng.choice(["bf16", "bf16", "bf16", "fp32"])
        r = _spread(rng, 24, 1280 if dtype == "bf16" else 400, tiles)
        s = _spread(rng, 8, 512, tiles)
        room = 20e12 if dtype == "bf16" else 1.5e12
        blocks = int(max(1, min(48, room / _block_flops(s, r))))
        return dict(path=path, dtype=dtype, blocks=blocks, n_seq=s, n_res=r, tail=tail, chunk=rng.choice([0, 0, 0, 64]))
    if path == "train":
        dtype = rng.choice(["bf16", "bf16", "fp32"])
        r = _spread(rng, 24, 512 if dtype == "bf16" else 256, tiles)
        s = _spread(rng, 8, 192, tiles)
        blocks = int(max(1, min(4, (2e12 if dtype == "bf16" else 4e11) / _block_flops(s, r))))
        return dict(path=path, dtype=dtype, blocks=blocks, n_seq=s, n_res=r, tail=tail)
    if path == "extra_msa":
        return dict(path=path, dtype="bf16", blocks=rng.choice([1, 4]), n_seq=_spread(rng, 64, 1536, tiles),
                    n_res=_spread(rng, 32, 640, tiles), tail=tail)
    if path == "template":
        return dict(path=path, dtype="bf16", blocks=2, n_templ=rng.randint(1, 4), n_res=_spread(rng, 32, 640, tiles), tail=tail)
    n, heads = _spread(rng, 24, 768, tiles), rng.choice([4, 8])
    most = max(1, min(512, int(1.2e8 / (heads * n * n))))
    return dict(path=path, dtype=rng.choice(["bf16", "bf16", "fp32"]), b2=round(math.exp(rng.uniform(math.log(max(1, most / 8)), math.log(most)))),
                heads=heads, n=n)


# ------------------------------------------------------------------------------------------------ preparation ----
_MODELS = {}      # what a program keeps loaded; a few at a time


def _model(key, build, dtype):
    if key not in _MODELS:
        while len(_MODELS) >= 4:
            _MODELS.pop(next(iter(_MODELS)))
        with torch.device("cuda"):
            mod = build()
        g = torch.Generator(device="cuda").manual_seed(0)
        with torch.no_grad():
            for name, p in mod.named_parameters():
                p.normal_(0.0, 0.02, generator=g)
                if "norm" in name and name.endswith("weight"):
                    p.add_(1.0)
        _MODELS[key] = mod.to(dtype)
    return _MODELS[key]


def _residue_mask(r, tail, dtype):
    mask = torch.ones(r, device="cuda", dtype=dtype)
    n = int(round(tail * r))
    if n:
        mask[r - n:] = 0
    return mask


def prepare(case, seed):
    dt = DTYPES[case["dtype"]]
    g = torch.Generator(device="cuda").manual_seed(seed)

    def normal(*shape):
        return torch.randn(*shape, device="cuda", dtype=dt, generator=g)

    path = case["path"]
    st = dict(path=path, seed=seed)
    if path == "kernels":
        b2, h, n = case["b2"], case["heads"], case["n"]
        mask = (torch.rand(1, b2, n, device="cuda", generator=g) > 0.1).to(dt)
        mask[..., 0] = 1
        st.update(mask=mask, logits=normal(1, b2, h, n, n), bias=normal(1, 1, h, n, n), d_probs=normal(1, b2, h, n, n),
                  x=normal(b2, n, h * 32), d_norm=normal(b2, n, h * 32), q=normal(1, b2, h, n, 32), k=normal(1, b2, h, n, 32),
                  v=normal(1, b2, h, n, 32), pair_bias=normal(1, h, n, n), d_att=normal(1, b2, n, h * 32),
                  norm=_model(("norm", h, dt), lambda: LayerNorm(h * 32), dt))
        for k in ("logits", "bias", "x", "q", "k", "v", "pair_bias"):
            st[k].requires_grad_(True)
        return st
    r = case["n_res"]
    res = _residue_mask(r, case["tail"], dt)
    st["pair_mask"] = res[:, None] * res[None, :]
    if path == "template":
        st["t"] = normal(case["n_templ"], r, r, C_T)
        st["z"] = normal(r, r, C_Z)
        st["pair_mask"] = st["pair_mask"][None]
        st["template_mask"] = torch.ones(case["n_templ"], device="cuda", dtype=dt)
        st["stack"] = _model(("template", case["blocks"], dt), lambda: TemplatePairStack(
            c_t=C_T, c_hidden_tri_att=16, c_hidden_tri_mul=64, no_blocks=case["blocks"], no_heads=4, pair_transition_n=2,
            dropout_rate=0.25, blocks_per_ckpt=None).eval(), dt)
        st["pointwise"] = _model(("pointwise", dt), lambda: TemplatePointwiseAttention(
            c_t=C_T, c_z=C_Z, c_hidden=16, no_heads=4, inf=1e5).eval(), dt)
        return st
    s = case["n_seq"]
    st["msa_mask"] = torch.ones(s, 1, device="cuda", dtype=dt) * res[None, :]
    if path == "extra_msa":
        st["m"], st["z"] = normal(s, r, C_E), normal(r, r, C_Z)
        st["stack"] = _model((path, case["blocks"], dt),
                             lambda: ExtraMSAStack(c_m=C_E, c_z=C_Z, no_blocks=case["blocks"]).eval(), dt)
        return st
    train = path == "train"
    st["m"], st["z"] = normal(s, r, C_M), normal(r, r, C_Z)
    st["chunk"] = case.get("chunk", 0)
    st["stack"] = _model((path, case["blocks"], dt), lambda: EvoformerStack(
        c_m=C_M, c_z=C_Z, c_s=C_S, no_blocks=case["blocks"], blocks_per_ckpt=1).train(train), dt)
    if train:
        st["m"].requires_grad_(True)
        st["z"].requires_grad_(True)
        st["grads"] = (normal(s, r, C_M), normal(r, r, C_Z), normal(r, C_S))     # what the heads send back
    return st


# -------------------------------------------------------------------------------------------------------- one pass ----
def run(st):
    path = st["path"]
    if path == "trunk":
        with torch.no_grad():
            if st["chunk"]:
                set_chunk_size(st["chunk"])
                try:
                    m, z, s = st["stack"].inplace([st["m"]], [st["z"]], st["msa_mask"], st["pair_mask"], chunk_size=st["chunk"])
                finally:
                    set_chunk_size(None)
                return m[0], z[0], s
            return st["stack"](st["m"], st["z"], st["msa_mask"], st["pair_mask"], chunk_size=None)
    if path == "train":
        params = list(st["stack"].parameters())
        for p in params:
            p.grad = None
        st["m"].grad = st["z"].grad = None
        torch.manual_seed(st["seed"])                       # a reproducible run fixes its dropout
        out = st["stack"](st["m"], st["z"], st["msa_mask"], st["pair_mask"], chunk_size=None)
        torch.autograd.backward(out, st["grads"])
        # one flat buffer, as optimizers and gradient reductions take it
        flat = torch.cat([p.grad.reshape(-1) for p in params])
        return [t.detach() for t in out] + [st["m"].grad, st["z"].grad, flat]
    if path == "extra_msa":
        with torch.no_grad():
            return st["stack"](st["m"], st["z"], chunk_size=None, msa_mask=st["msa_mask"], pair_mask=st["pair_mask"])
    if path == "template":
        with torch.no_grad():
            t = st["stack"](st["t"], st["pair_mask"], chunk_size=None)
            return t, st["pointwise"](t, st["z"], template_mask=st["template_mask"])
    norm = st["norm"]
    probs = fused_softmax(st["logits"], st["mask"], st["bias"])
    y = norm(st["x"])
    o = fused_attention_core(st["q"], st["k"], st["v"], st["mask"], st["pair_bias"])
    grads = torch.autograd.grad((probs, y, o), (st["logits"], st["bias"], st["x"], norm.weight, norm.bias, st["q"], st["k"],
                                                st["v"], st["pair_bias"]), (st["d_probs"], st["d_norm"], st["d_att"]))
    return [probs.detach(), y.detach(), o.detach()] + list(grads)


# ------------------------------------------------------------------------------------------------------- accounting ----
def _tri_att_flops(r, c, heads, d):
    return 2 * r * r * c * (5 * heads * d + heads) + 4 * r * heads * r * r * d


def _tri_mul_flops(r, c, hidden):
    return 2 * r * r * c * (4 * hidden + c) + 2 * r * r * hidden * c + 2 * hidden * r ** 3


def _pair_flops(r):
    return 2 * _tri_mul_flops(r, C_Z, 128) + 2 * _tri_att_flops(r, C_Z, 4, 32) + 4 * r * r * C_Z * 4 * C_Z


def _opm_flops(s, r, c_m):
    return 4 * s * r * c_m * 32 + 2 * r * r * s * 1024 + 2 * r * r * 1024 * C_Z


def _block_flops(s, r):
    """One Evoformer block: 2 M N K per contraction."""
    proj = 2 * s * r * C_M * 5 * 256
    row = proj + 2 * r * r * C_Z * 8 + 4 * s * 8 * r * r * 32
    col = proj + 4 * r * 8 * s * s * 32
    return row + col + 4 * s * r * C_M * 4 * C_M + _opm_flops(s, r, C_M) + _pair_flops(r)


def _extra_block_flops(s, r):
    row = 2 * s * r * C_E * 5 * 64 + 2 * r * r * C_Z * 8 + 4 * s * 8 * r * r * 8
    col = 2 * s * r * C_E * (2 * 64 + 2 * 8) + 4 * r * 8 * s * 8
    return row + col + 4 * s * r * C_E * 4 * C_E + _opm_flops(s, r, C_E) + _pair_flops(r)


def work(case):
    es, path = BYTES[case["dtype"]], case["path"]
    if path == "kernels":
        b2, h, n = case["b2"], case["heads"], case["n"]
        logits, tokens = b2 * h * n * n, b2 * n * h * 32
        # softmax: x, dy in, y, dx out; LayerNorm: x, dy, y, dx; attention: q, k, v, do in, o, dq, dk, dv out; bias and d(bias) twice
        return {"bytes": es * (4 * logits + 4 * tokens + 8 * tokens + 4 * h * n * n + b2 * n),
                "flops": (4 + 10) * b2 * h * n * n * 32}
    r = case["n_res"]
    if path == "template":
        nt = case["n_templ"]
        block = 2 * _tri_mul_flops(r, C_T, 64) + 2 * _tri_att_flops(r, C_T, 4, 16) + 4 * r * r * C_T * 2 * C_T
        point = 2 * r * r * (C_Z * 64 * 2 + nt * C_T * 128) + 4 * nt * r * r * 64
        return {"bytes": es * r * r * (2 * nt * C_T + 2 * C_Z), "flops": nt * case["blocks"] * block + point}
    s, blocks = case["n_seq"], case["blocks"]
    if path == "extra_msa":
        return {"bytes": es * (s * r * C_E + 2 * r * r * C_Z + blocks * 0.8e6), "flops": blocks * _extra_block_flops(s, r)}
    tensors, weights = s * r * C_M + r * r * C_Z, blocks * 1.8e6
    if path == "train":      # outputs and input gradients beside the inputs and cotangents; a backward pass is two products per product
        return {"bytes": es * (4 * tensors + 2 * weights), "flops": 3 * blocks * _block_flops(s, r)}
    return {"bytes": es * (2 * tensors + weights), "flops": blocks * _block_flops(s, r)}


def tolerance(case):
    path = case["path"]
    if case["dtype"] == "bf16":
        if path == "train":
            # ReLU derivatives of hidden values within a rounding of zero go either way: a few per cent of the gradients behind them
            return {"rel": 0.03}
        # every update is rounded to bf16; 48 blocks of them accumulate
        return {"rel": 0.02 if case.get("blocks", 1) > 8 else 0.01}
    if path == "train":
        return {"rel": 1e-3}      # as above, with the rounding of 32-bit sums
    return {"rel": 2e-5}
