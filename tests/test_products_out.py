"""Which ``out`` the kernel API writes without a scratch tensor: never one whose
memory an operand reaches into, however the two tensors came to share it. And
which operands it hands on uncopied: no bf16 one off a 16-byte boundary."""

from __future__ import annotations

import pytest
import torch

from himuon_amd.kernels import _padded, _result, _span

M = 128
SHAPE = (1, M, M)


def _aligned(n):
    """n fp32 elements from a 64-byte boundary on, with room on both sides."""
    buf = torch.zeros(n + 96)
    k = (-buf.data_ptr() % 64) // 4 + 32
    return buf[k: k + n]


@pytest.mark.parametrize("shift", [0, 4, M, M * M - 4, M * M, 2 * M * M])
@pytest.mark.parametrize("front", [True, False])
@pytest.mark.parametrize("imported", [True, False], ids=["dlpack", "view"])
def test_memory_that_an_operand_reaches_into_is_not_written(shift, front, imported):
    buf = _aligned(3 * M * M)
    one, two = buf[: M * M].view(SHAPE), buf[shift: shift + M * M].view(SHAPE)
    out, operand = (one, two) if front else (two, one)
    if imported:  # a storage of its own over the same memory
        out = torch.from_dlpack(out)
        assert shift == 0 or out.untyped_storage().data_ptr() != operand.untyped_storage().data_ptr()
    other = _aligned(M * M).view(SHAPE)
    got = _result(out, SHAPE, other, operand)
    assert (got is out) if shift >= M * M else (got is None)


def test_a_strided_operand_around_out():
    wide = _aligned(2 * M * M).view(1, M, 2 * M)  # its rows lie on both sides of out's
    out = torch.from_dlpack(wide.view(2, M, M)[1:])
    assert _result(out, SHAPE, wide[..., :M]) is None
    assert _span(wide[..., :M])[1] - wide.data_ptr() == 4 * (2 * M * M - M)
    assert _span(torch.empty(0, M, M)) == (0, 0)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("off", [0, 1, 4, 8])
def test_operands_handed_to_the_kernels(dtype, off):
    t = _aligned(M * M + 8).to(dtype)
    t = t[-t.data_ptr() % 16 // t.element_size():][off: off + 64 * 128].view(1, 64, 128).normal_()
    got = _padded(t, 64, 128)
    assert torch.equal(got, t) and (got is t) == (dtype == torch.float32 or off % 8 == 0)
    assert dtype == torch.float32 or got.data_ptr() % 16 == 0
