"""The block sizes of the products: 64 x 64, 128 x 128 and, for bf16, 256 x 256
output blocks, chosen by size and dtypes, one result."""

from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu

if torch.cuda.is_available():
    from himuon_amd import _native as nat

DEV = "cuda"


@pytest.mark.parametrize("idt,odt,B,M,N", [
    ("float16", torch.float32, 64, 1024, 1024), ("bfloat16", torch.float32, 8, 2048, 2048),
    ("float16", torch.float16, 32, 512, 16384), ("float8_e5m2", torch.float16, 64, 1024, 4096),
    ("bfloat16", torch.float16, 4, 4096, 2048)])
def test_block_sizes_give_the_same_bits(idt, odt, B, M, N):
    """Batches of long contractions, on 128 x 128 blocks where one matrix alone is
    on 64 x 64 blocks (which of the three products change is the dtypes'): bit for
    bit the same."""
    g = torch.Generator(device=DEV).manual_seed(M + N)
    dt = getattr(torch, idt)
    x = (torch.randn(B, M, N, device=DEV, generator=g) / N ** 0.5).to(dt)
    s = (torch.randn(B, M, M, device=DEV, generator=g) / M ** 0.5).to(dt)
    for shape, call in (((M, M), lambda i, o: nat.xxt_typed(x[i], o, o.shape[0], M, N)),
                        ((M, M), lambda i, o: nat.ba_plus_caa_typed(s[i], o, o.shape[0], M, 0.5, -1.5)),
                        ((M, N), lambda i, o: nat.bmm_add_typed(s[i], x[i], o, o.shape[0], M, N, 2.0))):
        whole, one = torch.empty(B, *shape, device=DEV, dtype=odt), torch.empty(1, *shape, device=DEV, dtype=odt)
        call(slice(0, B), whole)
        for k in range(0, B, max(1, B // 4)):
            call(slice(k, k + 1), one)
            assert torch.equal(one[0], whole[k])


@pytest.mark.parametrize("B,M,N", [(269, 256, 256), (198, 512, 512), (13, 1024, 1024), (17, 1024, 1024), (50, 1024, 1024),
                                   (2, 2560, 2560), (2, 3072, 6144), (1, 5120, 5120)])
def test_bf16_block_choice(B, M, N):
    """On either side of the lines between the 256 x 256 blocks and the smaller
    ones (himuon_xxt, himuon_ba_plus_caa, himuon_bmm_add): the smaller blocks' bits."""
    g = torch.Generator(device=DEV).manual_seed(M + N)
    x = (torch.randn(B, M, N, device=DEV, generator=g) / N ** 0.5).bfloat16()
    s = torch.randn(B, M, M, device=DEV, generator=g) / M ** 0.5
    s = (s + s.transpose(1, 2)).bfloat16().contiguous()  # (ba_plus_cAA's operand is symmetric)
    for shape, call in (((B, M, M), lambda o, f: nat.xxt(x, o, B, M, N, family=f)),
                        ((B, M, M), lambda o, f: nat.ba_plus_caa(s, o, B, M, 0.5, -1.5, family=f)),
                        ((B, M, N), lambda o, f: nat.bmm_add(s, x, o, B, M, N, 2.0, family=f))):
        a, b = (torch.empty(shape, device=DEV, dtype=torch.bfloat16) for _ in range(2))
        call(a, "auto"), call(b, "block128")
        assert torch.equal(a, b)
