"""The three NS products on 64 x 64 and 128 x 128 blocks (ns5_blk.hip) at the
edges of their range: two K units only, one block, odd block counts, row counts that are
no multiple of 256, more blocks than fit the chip at once. Each against float64
within a bound from the roundings it makes (torch's own bf16 products split the
contraction for some of these shapes, so equal bits are not the measure here):
half a bf16 ulp (at most 2^-8, eight significant bits) of every rounded value, and K 2^-24 of the sum of the
absolute products for the fp32 accumulation. And the choice of the block size
(ns_product): whatever it picks gives the bits of the 256 x 256 blocks."""

from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu

if torch.cuda.is_available():
    from himuon_amd import _native as nat
    from himuon_amd.engine import newton_schulz

DEV = "cuda"


@pytest.mark.parametrize("batch,M,N", [(1, 128, 128), (5, 128, 1152), (3, 640, 128), (2, 896, 2432), (1, 1024, 256),
                                       (180, 384, 384), (1, 64 * 11 * 2, 128)])
@pytest.mark.parametrize("round_once", [False, True])
def test_blk_products(batch, M, N, round_once):
    g = torch.Generator().manual_seed(M + N)
    X = (torch.randn(batch, M, N, generator=g) / (M * N) ** 0.5).to(torch.bfloat16).to(DEV)
    A = torch.empty(batch, M, M, device=DEV, dtype=torch.bfloat16)
    B, Y = torch.empty_like(A), torch.empty_like(X)
    nat.xxt(X, A, batch, M, N, family="block128")
    nat.ba_plus_caa(A, B, batch, M, nat.NS_C, nat.NS_B, family="block128")
    nat.bmm_add(B, X, Y, batch, M, N, nat.NS_A, round_once=round_once, family="block128")
    assert torch.equal(A, A.transpose(1, 2)) and torch.equal(B, B.transpose(1, 2))
    x, a, b = X.double(), A.double(), B.double()
    ulp, acc = 2.0**-8, 2.0**-24

    def mm(p, q):
        return torch.bmm(p, q.contiguous())

    def close(got, exact, bound):
        over = ((got.double() - exact).abs() - bound * 1.001).max().item()
        assert over <= 0, over

    xt = x.transpose(1, 2)
    s = mm(x, xt)
    close(A, s, ulp * s.abs() + N * acc * mm(x.abs(), xt.abs()))
    s, e = mm(a, a), M * acc * mm(a.abs(), a.abs())
    r = nat.NS_C * s + nat.NS_B * a
    close(B, r, ulp * r.abs() + nat.NS_C * e + 2 * acc * (nat.NS_C * s.abs() + abs(nat.NS_B) * a.abs()))
    s, e = mm(b, x), M * acc * mm(b.abs(), x.abs())
    e = e if round_once else e + ulp * (s.abs() + e)
    r = s + nat.NS_A * x
    close(Y, r, ulp * (r.abs() + e) + e + 2 * acc * (s.abs() + nat.NS_A * x.abs()))


@pytest.mark.parametrize("shape", [(3, 512, 512), (20, 512, 512), (40, 512, 512), (1024, 1024), (9, 1024, 1280),
                                   (70, 256, 512), (300, 256, 768), (16, 512, 1024),
                                   (28, 1024, 1024), (50, 1024, 1024), (80, 1024, 1024),
                                   (2, 880, 1345), (1, 770, 768), (3, 2100, 700)],
                         ids=lambda s: "x".join(map(str, s)))
def test_block_size_choice_gives_the_256_blocks_bits(shape):
    """(From 768 rows on the choice also writes X0 first, which family stream3
    forms as the first iteration reads X.)"""
    G = (torch.randn(*shape, generator=torch.Generator().manual_seed(5)) * 1e-3).to(DEV)
    for steps in (1, 2):
        assert torch.equal(newton_schulz(G, steps=steps), newton_schulz(G, steps=steps, family="stream3"))
