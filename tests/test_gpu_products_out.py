"""The entry points of himuon_amd.kernels write an ``out`` of the kernels' own
shape directly and every other one through a scratch tensor; which one holds is
not visible: the same bits in a contiguous ``out``, in a view at an odd element
offset, in every other column of a wider tensor, and in an ``out`` that shares
the operands' storage. Sizes: one 128 block and an edge of one 64 block and
several batches."""

from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu

if torch.cuda.is_available():
    from himuon_amd import kernels as K

DEV = "cuda"
DTYPES = [torch.float32, torch.float16, torch.bfloat16]


def _calls(B, M, N, dtype):
    g = torch.Generator().manual_seed(M + N)
    x = (torch.randn(B, M, N, generator=g) / N ** 0.5).to(dtype).to(DEV)
    s = (torch.randn(B, M, M, generator=g) / M ** 0.5).to(dtype).to(DEV)
    s = (s + s.transpose(1, 2)).contiguous()
    return [((B, M, M), x, lambda o: K.XXT(x, o)),
            ((B, M, M), s, lambda o: K.ba_plus_cAA(s, 0.5, -1.5, o)),
            ((B, M, N), x, lambda o: K.fused_bmm_add(s, x, 2.0, o))]


@pytest.mark.parametrize("dtype", DTYPES, ids=str)
@pytest.mark.parametrize("B,M,N", [(1, 128, 128), (3, 128, 384), (2, 320, 200)])
def test_every_out_holds_the_same_bits(B, M, N, dtype):
    for shape, _, call in _calls(B, M, N, dtype):
        plain = torch.empty(shape, device=DEV, dtype=dtype)
        version = plain._version
        assert call(plain) is plain and plain._version > version
        flat = torch.full((plain.numel() + 2,), 7.0, device=DEV, dtype=dtype)
        odd = flat[1:-1].view(shape)
        assert torch.equal(call(odd), plain) and flat[0] == 7 and flat[-1] == 7
        wide = torch.full((*shape[:2], 2 * shape[2]), 7.0, device=DEV, dtype=dtype)
        assert torch.equal(call(wide[..., ::2]), plain) and bool((wide[..., 1::2] == 7).all())


@pytest.mark.parametrize("dtype", DTYPES, ids=str)
def test_out_in_the_operands_storage(dtype):
    for shape, operand, call in _calls(2, 128, 128, dtype):
        want = call(torch.empty(shape, device=DEV, dtype=dtype)).clone()
        assert torch.equal(call(operand), want)


@pytest.mark.parametrize("dtype", DTYPES, ids=str)
@pytest.mark.parametrize("shift", [0, 8, 64 * 128])
def test_out_over_an_operands_memory_with_a_storage_of_its_own(dtype, shift):
    shape, n = (2, 128, 128), 2 * 128 * 128
    g = torch.Generator().manual_seed(5)
    vals, b = ((torch.randn(shape, generator=g) / 128 ** 0.5).to(dtype).to(DEV) for _ in range(2))
    for call in (lambda x, o: K.XXT(x, o), lambda x, o: K.ba_plus_cAA(x, 0.5, -1.5, o),
                 lambda x, o: K.fused_bmm_add(b, x, 2.0, o), lambda x, o: K.fused_bmm_add(x, b, 2.0, o)):
        want = call(vals, torch.empty_like(vals))
        buf = torch.zeros(64 + n + shift, device=DEV, dtype=dtype)
        x, out = buf[64: 64 + n].view(shape), torch.from_dlpack(buf[64 + shift: 64 + shift + n]).view(shape)
        assert out.untyped_storage().data_ptr() != x.untyped_storage().data_ptr()
        x.copy_(vals)
        assert torch.equal(call(x, out), want)


def test_out_that_requires_grad_and_inference_out_are_refused_as_before():
    shape, _, call = _calls(1, 128, 128, torch.float32)[0]
    with pytest.raises(RuntimeError):
        call(torch.empty(shape, device=DEV, requires_grad=True))
    with torch.inference_mode():
        o = torch.empty(shape, device=DEV)
        call(o)
    with pytest.raises(RuntimeError):
        call(o)
