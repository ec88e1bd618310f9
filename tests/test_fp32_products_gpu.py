"""fp32 products as six products of bf16 parts (ffk_fused_linear, ffk_bgemm_nt and ffk_weight_grad in fp32) against float64: error bounds, edges of
the tiles, infinite and undefined operands."""
import pytest
import torch

pytestmark = pytest.mark.gpu
INF = float("inf")


def _run(x, w):
    from fastfold_amd import _lib
    from fastfold_amd.model.fastnn import _fused as F_
    (M, K), N = x.shape, w.shape[0]
    o = torch.empty(M, N, device=x.device)
    if K in (128, 256):
        F_.linear(x, torch.cat([w, w.new_zeros((-N) % 128, K)]), None, N, out=o)
    else:
        _lib.bgemm_nt(x, w, o, M=M, N=N, K=K, lda=K, ldb=K, s_i=N)
    return o.double()


# every kernel of the two entry points: one slab of 32 or 64 rows and persistent workgroups; tiles of 32, 64 and 128; K that ends
# inside a step of 16, and the quarters of K
SHAPES = [(M, 128, N) for M in (1, 33, 1000) for N in (32, 36, 512)] + [(13689, 128, 512), (20001, 128, 128)] \
    + [(M, 256, N) for M in (1, 65, 4097) for N in (64, 256)] + [(8200, 256, 1024)] \
    + [(1, 36, 4), (63, 20, 33), (129, 64, 65), (4000, 40, 300), (33, 512, 128), (300, 1024, 100), (16400, 512, 128), (30000, 1024, 129)]


@pytest.mark.parametrize("M,K,N", SHAPES)
@pytest.mark.parametrize("sx,sw", [(1.0, 1.0), (1e-25, 1e20)])
def test_error_of_products(dev, M, K, N, sx, sw):
    g = torch.Generator().manual_seed(M + K + N)
    x, w = (torch.randn(M, K, generator=g) * sx).to(dev), (torch.randn(N, K, generator=g) * sw).to(dev)
    got, want, size = _run(x, w), x.double() @ w.double().t(), x.double().abs() @ w.double().abs().t()
    # what is left out of a product: x2 y3 + x3 y2 + x3 y3, at most 2^-24 (1 + 2^-10) of it (tests/test_fp32_parts.py); roundings of the sum:
    # six for a step of 16 and three for the pieces, each at most 2^-23 (cut off) of the sums of magnitudes
    err = (got - want).abs()
    assert bool((err <= (1 + 6 * ((K + 15) // 16) + 3) * 2.0 ** -23 * size).all())
    # independent roundings add up as a random walk: at most what one rounding of 2^-24 for every product of the sum would give
    assert float(err.norm() / want.norm()) <= max(K, 32) ** 0.5 * 2.0 ** -24


@pytest.mark.parametrize("K", [4, 128, 256])
def test_error_of_single_products(dev, K):
    """Every product by itself, over two million pairs of mantissas: what is left out of one (2^-24 (1 + 2^-10)) and the sum's cutting off of
    the terms below its last place (2^-23 for the largest of them, 2^-30 for those below 2^-7)."""
    g = torch.Generator().manual_seed(K)
    x, w = torch.zeros(2048, K), torch.zeros(1024, K)
    x[:, K // 2], w[:, K // 2] = (1 + torch.rand(n, generator=g) for n in (2048, 1024))
    # the mantissas whose parts are as large as they get, among them those of a first part that is cut off
    x[:4, K // 2] = w[:4, K // 2] = torch.tensor([0x3F80FEFF, 0x3F807F7F, 0x3F80FF7F, 0x3F8080FF], dtype=torch.int32).view(torch.float32)
    got, want = _run(x.to(dev), w.to(dev)).cpu(), x.double() @ w.double().t()
    assert float(((got - want) / want).abs().max()) <= 2.0 ** -24 * (1 + 2.0 ** -10) + 2.0 ** -23 + 2.0 ** -28


@pytest.mark.parametrize("M,K,N", [(100, 128, 256), (40000, 128, 512), (100, 256, 256), (20000, 256, 256), (300, 64, 64), (300, 1024, 128)])
def test_operands_that_round_to_infinity_are_finite(dev, M, K, N):
    """Numbers between the largest bf16 number and the largest fp32 number, on either side."""
    g = torch.Generator().manual_seed(M)
    x, w = torch.randn(M, K, generator=g), torch.randn(N, K, generator=g) * 2.0 ** -20
    top = torch.finfo(torch.float32).max
    x[3, 5], x[M // 2, 1], x[M - 1, 0] = top, -top, top * (1 - 2.0 ** -9)
    w[7], x[:, 2], w[:, 2] = 0.0, 0.0, 0.0
    x[M // 3, 2], w[7, 2] = 2.0 ** -20, -top
    x, w = x.to(dev), w.to(dev)
    got, want = _run(x, w), x.double() @ w.double().t()
    assert bool(got.isfinite().all())
    assert bool(((got - want).abs().amax(1) <= K ** 0.5 * 2.0 ** -23 * want.abs().amax(1) + 1e-30).all())


@pytest.mark.parametrize("M,K,N", [(100, 128, 256), (5000, 128, 512), (40000, 128, 512), (100, 256, 256), (20000, 256, 1024),
                                   (300, 1024, 128), (30000, 512, 128), (300, 64, 64), (3000, 64, 300)])
def test_infinite_and_undefined_operands(dev, M, K, N):
    g = torch.Generator().manual_seed(M + K + N)
    x, w = torch.randn(M, K, generator=g), torch.randn(N, K, generator=g)
    x[3, 5], x[M // 2, 1], x[M - 1, 0], w[7, 9], w[N - 1, 5] = INF, -INF, float("nan"), INF, -INF
    x, w = x.to(dev), w.to(dev)
    got, want = _run(x, w), x.double() @ w.double().t()
    assert torch.equal(got.isnan(), want.isnan())
    inf = want.isinf()
    assert torch.equal(got[inf], want[inf]) and bool(got[want.isfinite()].isfinite().all())
    ok = want.isfinite()
    assert float((got[ok] - want[ok]).norm() / want[ok].norm()) <= max(K, 32) ** 0.5 * 2.0 ** -24


@pytest.mark.parametrize("M,K,N", [(100, 128, 256), (5000, 128, 512), (40000, 128, 512), (100, 256, 256), (20000, 256, 1024),
                                   (300, 1024, 128), (30000, 512, 128), (300, 64, 64), (3000, 64, 300)])
def test_other_sums_keep_their_bits(dev, M, K, N):
    """Infinite and undefined operands change the sums they belong to and no others."""
    g = torch.Generator().manual_seed(M + K)
    x, w = torch.randn(M, K, generator=g).to(dev), torch.randn(N, K, generator=g).to(dev)
    clean = _run(x, w)
    rows, cols = [3, M // 2, M - 1], [7, N - 1]
    x[3, 5], x[M // 2, 1], x[M - 1, 0], w[7, 9], w[N - 1, 5] = INF, -INF, float("nan"), INF, -INF
    got = _run(x, w)
    clean[rows] = got[rows] = 0.0
    clean[:, cols] = got[:, cols] = 0.0
    assert torch.equal(got, clean)


def test_single_products_are_rounded_once(dev):
    """Sums of so few products are taken by the fp32 instructions: one product alone is the fp32 product."""
    from fastfold_amd import _lib
    g = torch.Generator().manual_seed(3)
    x, w = torch.zeros(300, 4), torch.zeros(200, 4)
    x[:, 2], w[:, 2] = torch.randn(300, generator=g), torch.randn(200, generator=g)
    assert torch.equal(_run(x.to(dev), w.to(dev)).float().cpu(), x[:, 2, None] * w[None, :, 2])
    for M in (1, 2):
        y, x = torch.randn(M, 136, generator=g), torch.randn(M, 40, generator=g)
        y[1:], x[1:] = 0.0, 0.0
        ws, out, cs = torch.empty(136 * 41, device=dev), torch.empty(136, 40, device=dev), torch.empty(136, device=dev)
        _lib.weight_grad(out, cs, ws, y.to(dev), x.to(dev), M=M, N=136, K=40, slices=1, dtype=torch.float32, y_map=(M, 0, 136), x_map=(M, 0, 40))
        assert torch.equal(out.cpu(), y[0, :, None] * x[0, None]) and torch.equal(cs.cpu(), y[0])


@pytest.mark.parametrize("M,K,N", [(40, 2048, 100), (700, 4096, 300), (4000, 4112, 2100), (64, 16384, 40)])
def test_long_sums_of_one_sign(dev, M, K, N):
    """What the instructions cut off has the sign of the sum: pieces of 256 with turned signs keep it from adding up."""
    g = torch.Generator().manual_seed(K)
    x, w = torch.rand(M, K, generator=g).to(dev), torch.rand(N, K, generator=g).to(dev)
    got, want = _run(x, w), x.double() @ w.double().t()
    # one rounding of the sum per piece of 256, at most 2^-24 of it each, adding up as a random walk, and 2^-23 for a piece's own products
    assert float((got - want).norm() / want.norm()) <= (K / 256) ** 0.5 * 2.0 ** -24 + 2.0 ** -23


@pytest.mark.parametrize("one_sign", [False, True])
@pytest.mark.parametrize("M,slices", [(31, 1), (256, 1), (257, 1), (600, 1), (5000, 3), (65536, 64), (65536, 1024)])
def test_error_of_weight_gradients(dev, M, slices, one_sign):
    from fastfold_amd import _lib
    g, N, K = torch.Generator().manual_seed(M), 136, 40
    y, x = ((torch.rand(M, C, generator=g) if one_sign else torch.randn(M, C, generator=g)).to(dev) for C in (N, K))
    ws, out, cs = torch.empty(slices * N * (K + 1), device=dev), torch.empty(N, K, device=dev), torch.empty(N, device=dev)

    def run():
        _lib.weight_grad(out, cs, ws, y, x, M=M, N=N, K=K, slices=slices, dtype=torch.float32, y_map=(M, 0, N), x_map=(M, 0, K))
        return out.double().cpu(), y.double().cpu().t() @ x.double().cpu()
    got, want = run()
    rel = lambda a, b: float((a - b).norm() / b.norm())
    # as above; the sums over the slices add slices / 4 + 3 roundings
    walk = (max(M / slices, 256) / 256 + slices / 4 + 3) ** 0.5 * 2.0 ** -24 + 2.0 ** -23
    assert rel(got, want) <= (walk if one_sign else 16 * 2.0 ** -24 + walk)       # of both signs: a piece's roundings against a sum that stays small
    assert rel(cs.double(), y.double().sum(0)) <= (M / slices + slices) ** 0.5 * 2.0 ** -24
    clean = got
    y[M // 2, 5], x[M // 3, 7], x[0, 9] = INF, -INF, float("nan")
    got, want = run()
    keep = torch.ones_like(clean, dtype=torch.bool)
    keep[5], keep[:, 7], keep[:, 9] = False, False, False
    assert torch.equal(got[keep], clean[keep])                # the other sums keep their bits
    fin = want.isfinite()
    assert torch.equal(got.isnan(), want.isnan()) and torch.equal(got[want.isinf()], want[want.isinf()])
    assert rel(got[fin], want[fin]) <= (M / slices + slices) ** 0.5 * 2.0 ** -24
