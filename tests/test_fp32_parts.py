"""The cut of an fp32 number into three bf16 numbers that the fp32 products are made of, restated: what is left out of a product."""
import torch


def _parts(x):
    out = []
    for _ in range(3):
        p = x.bfloat16().float()
        out.append(p)
        x = x - p
    return out


def test_parts_of_every_mantissa():
    """All 2^23 of them: the parts are the number, the second at most 2^-8 and the third at most 2^-17 of the power of two below it - so
    x2 y3 + x3 y2 + x3 y3 is at most 2^-24 (1 + 2^-10) of x y."""
    for lo in range(0, 1 << 23, 1 << 21):
        x = (torch.arange(lo, lo + (1 << 21), dtype=torch.int32) + 0x3F800000).view(torch.float32)
        x1, x2, x3 = _parts(x)
        assert torch.equal(x1.double() + x2.double() + x3.double(), x.double())
        assert float(x2.abs().max()) <= 2.0 ** -8 and float(x3.abs().max()) <= 2.0 ** -17


def test_what_is_left_out_of_a_product():
    g = torch.Generator().manual_seed(0)
    x, y = (1 + torch.rand(1 << 21, generator=g) for _ in range(2))
    worst = torch.tensor([0x3F807F7F, 0x3F80FF7F, 0x3F8080FF, 0x3F807F80], dtype=torch.int32).view(torch.float32)
    x[:16], y[:16] = worst.repeat(4), worst.repeat_interleave(4)
    (x1, x2, x3), (y1, y2, y3) = ([p.double() for p in _parts(v)] for v in (x, y))
    kept = x1 * y3 + x3 * y1 + x2 * y2 + x1 * y2 + x2 * y1 + x1 * y1
    full = x.double() * y.double()
    left = ((full - kept) / full).abs()
    assert 2.0 ** -25 < float(left.max()) <= 2.0 ** -24 * (1 + 2.0 ** -10)
