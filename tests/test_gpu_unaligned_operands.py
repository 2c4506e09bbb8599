"""Product operands and NS buffers off 16-byte boundaries: the block kernels'
direct-to-LDS loads do not take them, so the kernel API copies bf16 operands and
the C entry points run the register-staged kernels. The same bits as on aligned
memory, for every operand dtype, block family and rounding form; shapes of one
block, of whole and partial 256-blocks, of the fused pair and of X0 written first."""

from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu

if torch.cuda.is_available():
    from himuon_amd import _native as nat
    from himuon_amd import kernels as K

DEV = "cuda"
BF16 = torch.bfloat16


def _off(t, k):
    """t's values in contiguous memory k elements behind a 256-byte boundary."""
    buf = torch.empty(t.numel() + k, device=DEV, dtype=t.dtype)
    out = buf[k:].view(t.shape)
    out.copy_(t)
    assert out.data_ptr() % 16 and out.is_contiguous()
    return out


def _operands(B, M, N, dtype):
    g = torch.Generator().manual_seed(M + N)
    x = (torch.randn(B, M, N, generator=g) / N ** 0.5).to(dtype).to(DEV)
    s = torch.randn(B, M, M, generator=g) / M ** 0.5
    return x, (s + s.transpose(1, 2)).to(dtype).to(DEV).contiguous()


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, BF16], ids=str)
@pytest.mark.parametrize("B,M,N", [(1, 128, 128), (3, 128, 384), (2, 256, 512), (1, 200, 320)])
def test_kernel_api(B, M, N, dtype):
    x, s = _operands(B, M, N, dtype)
    for k in (1, 3):
        xo, so = _off(x, k), _off(s, k)
        for shape, call in (((B, M, M), lambda x, s, o: K.XXT(x, o)),
                            ((B, M, M), lambda x, s, o: K.ba_plus_cAA(s, 0.5, -1.5, o)),
                            ((B, M, N), lambda x, s, o: K.fused_bmm_add(s, x, 2.0, o))):
            out = [torch.empty(shape, device=DEV, dtype=dtype) for _ in range(3)]
            call(x, s, out[0]), call(xo, so, out[1]), call(xo, s, out[2])
            assert torch.equal(out[0], out[1]) and torch.equal(out[0], out[2])


@pytest.mark.parametrize("family", ["auto", "block128"])
@pytest.mark.parametrize("B,M,N", [(1, 128, 128), (3, 128, 384), (40, 256, 512), (2, 512, 768)])
def test_entry_points(B, M, N, family):
    x, s = _operands(B, M, N, BF16)

    def run(x, s, off):
        sq, rect = ([torch.empty(shape, device=DEV, dtype=BF16) for _ in range(3)] for shape in ((B, M, M), (B, M, N)))
        if off:
            sq, rect = [_off(t, 5) for t in sq], [_off(t, 5) for t in rect]
        nat.xxt(x, sq[0], B, M, N, family=family)
        nat.ba_plus_caa(s, sq[1], B, M, 0.5, -1.5, family=family)
        for k, once in enumerate((False, True)):
            nat.bmm_add(s, x, rect[k], B, M, N, 2.0, round_once=once, family=family)
        return sq[:2] + rect[:2]

    for a, b in zip(run(x, s, False), run(_off(x, 1), _off(s, 7), True)):
        assert torch.equal(a, b)


@pytest.mark.parametrize("round_once", [False, True])
@pytest.mark.parametrize("family", ["auto", "block128", "stream3"])
@pytest.mark.parametrize("n,mp,np_", [(3, 128, 384), (5, 256, 512), (2, 512, 512), (20, 512, 512), (2, 768, 896)])
def test_ns5_buffers(n, mp, np_, family, round_once):
    g = torch.Generator().manual_seed(mp)
    x0 = torch.randn(n, mp, np_, generator=g).to(BF16).to(DEV)
    inv = 1 / x0.float().square().sum(dim=(1, 2)).sqrt()
    ws_bytes = nat.ns5_workspace_bytes(2, mp, np_)
    for steps in (1, 4):
        out = []
        for bx, by, bw in ((0, 0, 0), (1, 3, 0), (0, 0, 2), (0, 1, 0)):
            x, y = ((_off(x0, k) if k else x0.clone()) for k in (bx, by))
            ws = torch.empty(ws_bytes + 16, device=DEV, dtype=torch.uint8)[bw:]
            nat.ns5(x, y, inv, n, mp, np_, steps, ws, 2, family=family, round_once=round_once)
            out.append((x, y)[steps % 2])
        assert all(torch.equal(o, out[0]) for o in out[1:])
