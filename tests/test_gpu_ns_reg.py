"""NS5 of 256 x 256 NS tiles on the register-resident kernel (ns5_reg.hip):
bit-identical to torch's same-dtype NS5 (bf16 products, fp32 accumulation in
ascending k, one rounding per product) for full, padded and tall tiles, both
rounding forms of the third product, and every step count's buffer parity; and
the whole step in one launch (himuon_reg_step) bit-identical to the separate
gather, normaliser, NS and untile launches."""

from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu

if torch.cuda.is_available():
    from himuon_amd import _native as nat
    from himuon_amd.engine import newton_schulz

    from gpu_ref import ns5_torch_staged
    from test_gpu_lds_step import _groups_table, _pair

DEV = "cuda"


@pytest.mark.parametrize("shape", [(1, 256, 256), (300, 256, 256), (3, 129, 131), (2, 200, 256), (2, 255, 130), (250, 251)],
                         ids=lambda s: "x".join(map(str, s)))
@pytest.mark.parametrize("steps", [1, 2, 5])
def test_ns_256_bit_identical_to_torch(shape, steps):
    """(300 tiles: more than one per CU; 129 x 131: all but one row of the
    second half is padding; 255 x 130: tall; a 2-D input: rounded once.)"""
    G = (torch.randn(*shape, generator=torch.Generator().manual_seed(3)) * 1e-3).to(DEV)
    m, n = sorted(shape[-2:])
    P = torch.zeros(*shape[:-2], 256, 256, device=DEV)  # the reference on the padded tile: the same sums
    P[..., :m, :n] = G if shape[-2] <= shape[-1] else G.transpose(-2, -1)
    ref = ns5_torch_staged(P, steps=steps, round_once=len(shape) == 2)[..., :m, :n]
    ref = ref if shape[-2] <= shape[-1] else ref.transpose(-2, -1)
    out = newton_schulz(G, steps=steps)
    assert torch.equal(out, ref), (out - ref).norm() / ref.norm()


F32, BF16 = torch.float32, torch.bfloat16


@pytest.mark.parametrize("gdt,pdt", [(F32, F32), (F32, BF16), (BF16, BF16), (BF16, F32)])
@pytest.mark.parametrize("th,tw,steps,momentum,round_once", [
    (256, 256, 5, "nesterov", False), (256, 256, 2, "plain", True), (256, 256, 0, "nesterov", False),
    (130, 255, 1, "none", False)])
def test_reg_step_equals_the_four_launches(gdt, pdt, th, tw, steps, momentum, round_once):
    """Ragged edges, a parameter smaller than a tile, an unaligned row stride,
    two groups, two chunks (the second not at tile 0)."""
    shapes = [(600, 400), (256, 256), (512, 777), (77, 130)]
    pairs = _pair(shapes, th, tw, gdt, pdt, momentum == "nesterov", momentum != "none", round_once, steps)
    (p_sep, m_sep, g_sep), (p_fus, m_fus, g_fus) = pairs
    assert g_fus.reg_step_ok() and not g_fus.lds_step_ok()
    sa, n = _groups_table(), g_sep.n_tiles
    ws = torch.empty(nat.ns5_workspace_bytes(n, g_sep.mp, g_sep.np), device=DEV, dtype=torch.uint8)
    g_sep.gather()
    g_sep.ns(0, n, steps, ws, n)
    g_sep.untile(steps, sa)
    g_fus.reg_step(0, 5, steps, sa)
    g_fus.reg_step(5, n - 5, steps, sa)
    for a, b in zip(p_sep, p_fus):
        assert torch.equal(a, b)
    for a, b in zip(m_sep, m_fus):
        assert a is None or torch.equal(a, b)


def test_reg_step_refuses_other_buckets():
    args = [8, 1, 0, 0, 256, 256, 0, 1, 5, 1.0, 1.0, 1.0, 1e-7, 0x10, 16, None]
    assert nat.load().himuon_reg_step(*args) == 0  # empty work: no launch
    for pos, val in [(4, 128), (4, 257), (5, 255), (5, 512), (6, 2), (7, 2), (8, -1), (13, 1), (0, None), (14, None), (2, -1)]:
        bad = list(args)
        bad[pos] = val
        assert nat.load().himuon_reg_step(*bad) == -22, (pos, val)
