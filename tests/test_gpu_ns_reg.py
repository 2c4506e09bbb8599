"""NS5 of 256 x 256 NS tiles on the register-resident kernel (ns5_reg.hip):
bit-identical to torch's same-dtype NS5 (bf16 products, fp32 accumulation in
ascending k, one rounding per product) for full, padded and tall tiles, both
rounding forms of the third product, and every step count's buffer parity."""

from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu

if torch.cuda.is_available():
    from himuon_amd.engine import newton_schulz

    from gpu_ref import ns5_torch_staged

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
