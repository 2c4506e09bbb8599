"""Gather and untile of rows at any element alignment (odd widths, column
slices, storage offsets), whose vectors straddle 16-byte boundaries, and the
normaliser of tiles of many partials: bit-identical to the same data in aligned
rows, and to the sum of squares added in order."""

from __future__ import annotations

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

if torch.cuda.is_available():
    from himuon_amd import _native as nat
    from himuon_amd.engine import TileGroup

    from test_gpu_lds_step import _groups_table

DEV = "cuda"
F32, BF16, F16 = torch.float32, torch.bfloat16, torch.float16


def _at(t, pitch, offset):
    """t's values in rows of `pitch` elements starting `offset` elements into a buffer."""
    h, w = t.shape
    buf = torch.zeros(offset + h * pitch, device=DEV, dtype=t.dtype)
    v = buf[offset:].view(h, pitch)[:, :w]
    v.copy_(t)
    return v


@pytest.mark.parametrize("tile", [(512, 512), (256, 256), (128, 128), (300, 300), (512, 256)])
@pytest.mark.parametrize("gdt,pdt", [(F32, BF16), (BF16, BF16), (F32, F32), (F16, F16)])
def test_rows_at_any_alignment(tile, gdt, pdt):
    h, w = 701, 1003
    g = torch.Generator().manual_seed(4)
    p0, g0, m0 = ((torch.randn(h, w, generator=g) * s).to(DEV) for s in (0.02, 1e-3, 3e-3))
    sa, out = _groups_table(), []
    # rows of 1008 elements (a multiple of 16 bytes), of 1003 (odd), and of 1004 starting one element in
    for pitch, offset in ((1008, 0), (1003, 0), (1004, 1)):
        p, gr, m = _at(p0.to(pdt), pitch, offset), _at(g0.to(gdt), pitch, offset), _at(m0.to(gdt), pitch, offset)
        grp = TileGroup([p], [gr], [m], tile[0], tile[1], upd_scales=[4.5], mus=[0.95], nesterovs=[True],
                        device=torch.device(DEV), dtype=gdt, apply_groups=[1])
        step = grp.whole_step()
        if step:
            step(0, grp.n_tiles, 5, sa)
        else:
            ws = torch.empty(grp.workspace_bytes(grp.n_tiles), device=DEV, dtype=torch.uint8)
            grp.gather()
            if grp.ns_untile_ok(5):
                grp.ns_untile(0, grp.n_tiles, 5, ws, grp.n_tiles, sa)
            else:
                grp.ns(0, grp.n_tiles, 5, ws, grp.n_tiles)
                grp.untile(5, sa)
        out.append((p.clone(), m.clone()))
    for p, m in out[1:]:
        assert torch.equal(p, out[0][0]) and torch.equal(m, out[0][1])


@pytest.mark.parametrize("per_tile", [1, 16, 17, 63, 64, 65, 768])
@pytest.mark.parametrize("n", [1, 5])
def test_tile_scale_adds_in_order(per_tile, n):
    x = torch.rand(n, per_tile, generator=torch.Generator().manual_seed(per_tile)) ** 4
    inv = torch.empty(n, device=DEV)
    nat.tile_scale(x.to(DEV), per_tile, n, inv)
    s = np.zeros(n, np.float32)
    for q in range(per_tile):
        s = s + x.numpy()[:, q]
    exp = np.float32(1) / (np.sqrt(s) + np.float32(nat.NS_EPS))
    assert np.array_equal(inv.cpu().numpy(), exp)
