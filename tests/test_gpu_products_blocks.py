"""The block sizes of the typed products (himuon_*_typed): 128 x 128 output
blocks for long contractions of many blocks, 64 x 64 otherwise, one result."""

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
