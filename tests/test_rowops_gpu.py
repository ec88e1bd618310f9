"""GPU parity of the row-wise kernels through the C ABI, against the float64 numpy oracle.

Shapes, dtypes and tolerances follow the reference's own op tests
(tests/test_fastnn/test_softmax.py:7-38, tests/test_fastnn/test_layernorm.py:13-40)."""
import numpy as np
import pytest
import torch

from oracle import ops_np

pytestmark = pytest.mark.gpu

SOFTMAX_TOL = {torch.float32: 1e-6, torch.float16: 2e-4, torch.bfloat16: 1e-3}   # test_softmax.py:14
LN_TOL = {torch.float32: 1e-4, torch.float16: 1e-1, torch.bfloat16: 1e-1}        # test_layernorm.py:20


def _np(t):
    return t.detach().float().cpu().numpy().astype(np.float64)


@pytest.mark.parametrize("seq", [31, 32, 128, 129, 256, 259, 512, 700, 1024])
@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16])
def test_fused_softmax_reference_cases(dev, seq, dtype):
    from fastfold_amd.model.fastnn.kernel import fused_softmax
    g = torch.Generator().manual_seed(seq)
    x = torch.rand(1, 8, 4, seq, seq, generator=g).to(dev, dtype)
    mask = (torch.rand(1, 8, seq, generator=g) > 0.1).to(dev, dtype)
    mask[..., 0] = 1
    bias = torch.rand(1, 1, 4, seq, seq, generator=g).to(dev, dtype)
    for m_, b_ in ((mask, bias), (mask, None), (None, None)):
        out = fused_softmax(x, m_, b_) if b_ is not None else (fused_softmax(x, m_) if m_ is not None else fused_softmax(x))
        ref = ops_np.fused_softmax(_np(x), None if m_ is None else _np(m_), None if b_ is None else _np(b_))
        err = np.abs(_np(out) - ref).max()
        assert err < SOFTMAX_TOL[dtype], (seq, dtype, err)
        if m_ is not None and dtype == torch.float32:
            assert float(out[0, :, :, :, :][(m_[0] == 0)[:, None, None, :].expand_as(out[0])].abs().max()) == 0.0


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("b1,b2,h,nq,cols", [(1, 3, 2, 5, 24), (2, 7, 1, 9, 33), (1, 40, 2, 6, 64), (1, 5, 3, 7, 77), (1, 4, 2, 3, 130),
                                             (1, 64, 4, 24, 24), (1, 33, 2, 8, 257), (1, 9, 1, 2, 770), (1, 2, 1, 3, 1023),
                                             (1, 3, 1, 2, 1025), (1, 2, 1, 2, 4104), (2, 3, 2, 4, 2048)])
def test_fused_softmax_rows_and_bias_gradient(dev, dtype, b1, b2, h, nq, cols):
    """Every access width of the row kernels (vectors, two elements, one element, rows beyond the register geometries), the
    bias gradient with one slice of the batch rows and with several, against float64 autograd of the formula."""
    from fastfold_amd.model.fastnn.kernel import fused_softmax
    g = torch.Generator().manual_seed(cols + b2)
    x = (2 * torch.randn(b1, b2, h, nq, cols, generator=g)).to(dev, dtype)
    mask = (torch.rand(b1, b2, cols, generator=g) > 0.2).to(dev, dtype)
    mask[..., 1] = 1
    bias = torch.randn(b1, 1, h, nq, cols, generator=g).to(dev, dtype)
    dy = torch.randn(b1, b2, h, nq, cols, generator=g).to(dev, dtype)
    xr, br = (t.double().cpu().requires_grad_(True) for t in (x, bias))
    ref = torch.softmax((xr + br).masked_fill(mask.cpu()[:, :, None, None, :] == 0, -1e9), -1)
    ref.backward(dy.double().cpu())
    xf, bf = x.clone().requires_grad_(True), bias.clone().requires_grad_(True)
    out = fused_softmax(xf, mask, bf)
    out.backward(dy)
    tol = {torch.float32: 2e-6, torch.bfloat16: 1e-2, torch.float16: 2e-3}[dtype]

    def rel(a, b):
        return float((a.detach().double().cpu() - b).norm() / b.norm())
    assert rel(out, ref.detach()) < tol
    assert rel(xf.grad, xr.grad) < 2 * tol and rel(bf.grad, br.grad) < 2 * tol
    xg = x.clone().requires_grad_(True)
    fused_softmax(xg, mask, bias).backward(dy)              # without a bias gradient
    assert rel(xg.grad, xr.grad) < 2 * tol


def test_fused_softmax_inplace_and_backward(dev):
    from fastfold_amd.model.fastnn.kernel import fused_softmax
    from fastfold_amd.model.fastnn.kernel.softmax import fused_softmax_
    g = torch.Generator().manual_seed(0)
    x = torch.randn(1, 5, 2, 40, 40, generator=g).to(dev)
    mask = (torch.rand(1, 5, 40, generator=g) > 0.2).float().to(dev)
    mask[..., 3] = 1
    bias = torch.randn(1, 1, 2, 40, 40, generator=g).to(dev)
    xr, br = x.clone().requires_grad_(True), bias.clone().requires_grad_(True)
    ref = torch.softmax(xr + br + 1e9 * (mask - 1)[:, :, None, None, :], -1)
    xf, bf = x.clone().requires_grad_(True), bias.clone().requires_grad_(True)
    out = fused_softmax(xf, mask, bf)
    assert (out - ref).abs().max().item() < 1e-6
    dy = torch.rand_like(out)
    ref.backward(dy)
    out.backward(dy)
    assert (xf.grad - xr.grad).abs().max().item() < 1e-6
    assert (bf.grad - br.grad).abs().max().item() < 1e-5
    y = x.clone()
    r = fused_softmax_(y, mask, bias)
    assert r.data_ptr() == y.data_ptr() and (y - ref.detach()).abs().max().item() < 1e-6


@pytest.mark.parametrize("shape", [(64, 64), (64, 128), (64, 129), (64, 1024), (3, 5, 256), (1000, 8)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16])
def test_layernorm_reference_cases(dev, shape, dtype):
    from fastfold_amd.model.fastnn.kernel import LayerNorm
    g = torch.Generator().manual_seed(shape[-1])
    x = torch.rand(*shape, generator=g).to(dev, dtype)
    ln = LayerNorm(shape[-1]).to(dev, dtype)
    with torch.no_grad():
        ln.weight.copy_(1 + 0.1 * torch.randn(shape[-1], generator=g))
        ln.bias.copy_(0.1 * torch.randn(shape[-1], generator=g))
    out = ln(x)
    ref = ops_np.layer_norm(_np(x), _np(ln.weight), _np(ln.bias), 1e-5)
    assert out.shape == x.shape and out.dtype == dtype
    assert np.abs(_np(out) - ref).max() < LN_TOL[dtype]
    if dtype == torch.float32:
        assert np.abs(_np(out) - ref).max() < 2e-6


def test_layernorm_backward(dev):
    from fastfold_amd.model.fastnn.kernel import LayerNorm
    g = torch.Generator().manual_seed(1)
    x = torch.randn(37, 129, generator=g).to(dev)
    ln = LayerNorm(129).to(dev)
    ref = torch.nn.LayerNorm(129).to(dev)
    with torch.no_grad():
        ln.weight.copy_(1 + 0.1 * torch.randn(129, generator=g))
        ref.weight.copy_(ln.weight)
    xa, xb = x.clone().requires_grad_(True), x.clone().requires_grad_(True)
    dy = torch.rand(37, 129, generator=g).to(dev)
    ln(xa).backward(dy)
    ref(xb).backward(dy)
    assert (xa.grad - xb.grad).abs().max().item() < 1e-4     # test_layernorm.py:20 (fp32)
    assert (ln.weight.grad - ref.weight.grad).abs().max().item() < 1e-4
    assert (ln.bias.grad - ref.bias.grad).abs().max().item() < 1e-4


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("rows,cols", [(65, 64), (1000, 128), (37, 256), (4096 + 3, 384), (513, 512), (70, 1024),
                                       (33, 2048), (40, 72)])
def test_layernorm_backward_shapes(dev, dtype, rows, cols):
    """Both backward kernels (the vector form for rows of exactly lanes x vectors x 16 bytes up to 1024 elements, the
    general one otherwise) against float64 autograd of torch's layer_norm on the same rounded inputs; row counts that
    leave ragged row groups, enough rows for several grid-stride passes."""
    from fastfold_amd.model.fastnn.kernel import LayerNorm
    g = torch.Generator().manual_seed(rows + cols)
    x = torch.randn(rows, cols, generator=g).to(dev, dtype)
    dy = torch.randn(rows, cols, generator=g).to(dev, dtype)
    ln = LayerNorm(cols).to(dev, dtype)
    with torch.no_grad():
        ln.weight.copy_(1 + 0.2 * torch.randn(cols, generator=g))
        ln.bias.copy_(0.1 * torch.randn(cols, generator=g))
    xa = x.clone().requires_grad_(True)
    ln(xa).backward(dy)
    xr = x.double().cpu().requires_grad_(True)
    wr, br = ln.weight.detach().double().cpu().requires_grad_(True), ln.bias.detach().double().cpu().requires_grad_(True)
    torch.nn.functional.layer_norm(xr, (cols,), wr, br, ln.eps).backward(dy.double().cpu())
    tol = 1e-5 if dtype == torch.float32 else (1.5e-2 if dtype == torch.bfloat16 else 2e-3)

    def rel(a, b):
        return float((a.double().cpu() - b).abs().max() / b.abs().max())
    assert rel(xa.grad, xr.grad) <= tol, rel(xa.grad, xr.grad)
    assert rel(ln.weight.grad, wr.grad) <= tol, rel(ln.weight.grad, wr.grad)
    assert rel(ln.bias.grad, br.grad) <= tol, rel(ln.bias.grad, br.grad)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("C", [128, 36, 7])
def test_elementwise_fusions(dev, dtype, C):
    from fastfold_amd.model.fastnn.kernel import bias_dropout_add, bias_sigmod_ele, bias_ele_dropout_residual
    g = torch.Generator().manual_seed(C)
    sh = (1, 6, 9, C)
    y, z, r = (torch.randn(*sh, generator=g).to(dev, dtype) for _ in range(3))
    b = torch.randn(C, generator=g).to(dev, dtype)
    tol = 1e-5 if dtype == torch.float32 else 4e-2
    out = bias_sigmod_ele(y, b, z)
    assert np.abs(_np(out) - ops_np.bias_sigmod_ele(_np(y), _np(b), _np(z))).max() < tol
    for dm in (torch.ones_like(y[:, 0:1, :, :]), torch.ones_like(y[:, :, 0:1, :])):
        dm = dm * 0.5   # any multiplier must be applied as given in eval mode
        out = bias_dropout_add(y, b, dm, r, prob=0.25, training=False)
        assert np.abs(_np(out) - ops_np.bias_dropout_add(_np(y), _np(b), _np(dm), _np(r))).max() < tol
        out = bias_ele_dropout_residual(y, b, z, dm, r, prob=0.25, training=False)
        assert np.abs(_np(out) - ops_np.bias_ele_dropout_residual(_np(y), _np(b), _np(z), _np(dm), _np(r))).max() < tol


def test_errors_raise_runtime_error(dev):
    from fastfold_amd.model.fastnn.kernel import fused_softmax
    with pytest.raises(RuntimeError):
        fused_softmax(torch.rand(2, 3, 4), torch.ones(2, 4))                       # CPU tensors
    x = torch.rand(1, 2, 2, 4, 4, device=dev)
    with pytest.raises(RuntimeError):
        fused_softmax(x, torch.ones(1, 2, 5, device=dev))                          # wrong mask shape
    with pytest.raises(RuntimeError):
        fused_softmax(x.double())                                                  # unsupported dtype


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("accesses", [1, 7, 8, 13, 16, 25, 32, 51, 64, 101, 128, 201, 256, 301, 512, 701])
def test_row_kernels_at_every_geometry(dev, dtype, accesses):
    """Rows of so many 16-byte, two-element and one-element accesses: the lanes and accesses per lane the row kernels are built
    with, whole and partly filled, forward and backward, against float64 on the GPU (one or two roundings to the type)."""
    from fastfold_amd.model.fastnn.kernel import LayerNorm, bias_dropout_add, bias_ele_dropout_residual, bias_sigmod_ele, fused_softmax
    vec = 4 if dtype == torch.float32 else 8
    tol = {torch.float32: 5e-6, torch.bfloat16: 1.5e-2, torch.float16: 2e-3}[dtype]
    g = torch.Generator(device=dev).manual_seed(accesses)

    def rnd(*s):
        return torch.randn(*s, device=dev, generator=g).to(dtype)

    def check(got, ref, what):
        for a, e in zip(got, ref):
            assert float(((a.double() - e).norm() / e.norm().clamp_min(1e-3)).detach()) <= tol, what
    for cols in {vec * accesses, 2 * accesses, accesses}:
        x, bias, dy = rnd(1, 3, 2, 5, cols).requires_grad_(True), rnd(1, 1, 2, 5, cols).requires_grad_(True), rnd(1, 3, 2, 5, cols)
        mask = (torch.rand(1, 3, cols, device=dev, generator=g) > 0.2).to(dtype)
        mask[..., -1] = 1
        xr, br = (t.detach().double().requires_grad_(True) for t in (x, bias))
        s = torch.where(mask[:, :, None, None] == 0, -1e9, xr + br).softmax(-1)
        ref = torch.autograd.grad(s, (xr, br), dy.double())
        y = fused_softmax(x, mask, bias)
        check((y, *torch.autograd.grad(y, (x, bias), dy)), (s, *ref), cols)
        check(torch.autograd.grad(fused_softmax(x, mask, bias.detach()), (x,), dy), ref[:1], cols)
        if cols == 1:
            continue                                     # a row of one element has no variance
        norm = LayerNorm(cols).to(dev, dtype)
        with torch.no_grad():
            norm.weight.copy_(1 + 0.2 * rnd(cols))
            norm.bias.copy_(0.1 * rnd(cols))
        x, dy = rnd(70, cols).requires_grad_(True), rnd(70, cols)
        xr, wr, br = (t.detach().double().requires_grad_(True) for t in (x, norm.weight, norm.bias))
        yr = torch.nn.functional.layer_norm(xr, (cols,), wr, br, norm.eps)
        y = norm(x)
        check((y, *torch.autograd.grad(y, (x, norm.weight, norm.bias), dy)), (yr, *torch.autograd.grad(yr, (xr, wr, br), dy.double())), cols)
        a, z, r, b, dm = rnd(1, 4, 3, cols), rnd(1, 4, 3, cols), rnd(1, 4, 3, cols), rnd(cols), rnd(1, 1, 3, cols)
        ad, zd, rd, bd, dd = (t.double() for t in (a, z, r, b, dm))
        check((bias_sigmod_ele(a, b, z), bias_dropout_add(a, b, dm, r, prob=0.25, training=False),
               bias_ele_dropout_residual(a, b, z, dm, r, prob=0.25, training=False)),
              (torch.sigmoid(ad + bd) * zd, rd + (ad + bd) * dd, rd + dd * (zd * (ad + bd))), cols)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("cols", [32, 64, 128, 256, 512])
def test_layernorm_bwd_entry_point(dev, dtype, cols):
    """ffk_layernorm_bwd at the lengths whose module goes to ffk_layernorm_bwd_rows: column sums by one atomic per column and block."""
    from fastfold_amd import _lib
    rows, g = 203, torch.Generator(device=dev).manual_seed(cols)
    x, dy, w = (torch.randn(*s, device=dev, generator=g).to(dtype) for s in ((rows, cols), (rows, cols), (cols,)))
    xr, wr, br = x.double().requires_grad_(True), w.double().requires_grad_(True), torch.zeros(cols, device=dev, dtype=torch.double).requires_grad_(True)
    ref = torch.autograd.grad(torch.nn.functional.layer_norm(xr, (cols,), wr, br), (xr, wr, br), dy.double())
    mean, rstd = x.float().mean(-1), (x.double().var(-1, unbiased=False) + 1e-5).rsqrt().float()
    dx, dw, db = torch.empty_like(x), torch.zeros(cols, device=dev), torch.zeros(cols, device=dev)
    _lib.call("ffk_layernorm_bwd", *(_lib.ptr(t) for t in (dx, dw, db, dy, x, mean, rstd, w)), rows, cols, _lib.dtype_tag(dtype), _lib.stream_ptr())
    for a, e, tol in zip((dx, dw, db), ref, ({torch.float32: 1e-5, torch.bfloat16: 1e-2, torch.float16: 2e-3}[dtype], 1e-5, 1e-5)):
        assert float((a.double() - e).norm() / e.norm()) <= tol
