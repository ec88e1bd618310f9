"""The weight layouts of the kernels that read fragments straight into registers, element by element (include/ffk.h)."""
import pytest
import torch

from fastfold_amd.model.fastnn import _fused as F_


@pytest.mark.parametrize("n,K", [(32, 16), (64, 96), (128, 32)])
def test_fragments_against_their_definition(n, K):
    w = torch.arange(n * K, dtype=torch.float32).view(n, K)
    plain = F_.pack_fragments(w, torch.float32, "cpu").view(n // 32, K // 16, 64, 8)
    acc = F_.pack_fragments_of_accumulators(w, torch.float32, "cpu").view(n // 32, K // 16, 64, 8)
    for b in range(n // 32):
        for s in range(K // 16):
            for lane in range(64):
                row, half = lane % 32, lane // 32
                tau = 16 * (row >> 2 & 1) + 4 * (row >> 3) + (row & 3)
                for e in range(8):
                    assert plain[b, s, lane, e] == w[32 * b + row, 16 * s + 8 * half + e]
                    assert acc[b, s, lane, e] == w[32 * b + tau, 16 * s + 8 * (e // 4) + 4 * half + e % 4]


@pytest.mark.parametrize("C", [64, 128, 256])
def test_attention_block_weights_are_five_of_one_size(C):
    g = torch.Generator().manual_seed(C)
    qkv, gate, out = (torch.randn(k * C, C, generator=g) for k in (3, 1, 1))
    w = F_.pack_attention_block(qkv, gate, out, torch.bfloat16, "cpu").view(5, C * C)
    for i, part in enumerate((*qkv.split(C), gate)):
        assert torch.equal(w[i], F_.pack_fragments(part, torch.bfloat16, "cpu"))
    assert torch.equal(w[4], F_.pack_fragments_of_accumulators(out, torch.bfloat16, "cpu"))


@pytest.mark.parametrize("C,hidden", [(64, 128), (64, 256), (128, 512)])
def test_transition_weights_against_their_definition(C, hidden):
    w1, w2 = (torch.randn(*n, generator=torch.Generator().manual_seed(C)).bfloat16() for n in ((hidden, C), (C, hidden)))
    p1, p2 = F_.pack_transition_block(w1, w2, torch.bfloat16, "cpu")
    lane = torch.arange(64)
    row, half = lane % 32, lane // 32
    sigma = 16 * (row >> 4) + 8 * (row >> 2 & 1) + 4 * (row >> 3 & 1) + (row & 3)
    tau = 16 * (row >> 2 & 1) + 4 * (row >> 3) + (row & 3)
    for w, p, perm in ((w1, p1, sigma), (w2, p2, tau)):
        n, K = w.shape
        p = p.view(n // 32, K // 16, 64, 8)
        for b in range(n // 32):
            for s in range(K // 16):
                assert torch.equal(p[b, s], w[(32 * b + perm)[:, None], 16 * s + 8 * half[:, None] + torch.arange(8)])
