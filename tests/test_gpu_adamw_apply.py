"""himuon_adamw_apply: the AdamW step with its WD/LR in the same pass leaves
moments, step counters and parameters bit-identical to himuon_adamw_step
followed by himuon_apply_updates, for every dtype pair, sizes around the
8-element vectors and the chunks, and two groups; and at the optimizer level
over steps with a changing learning rate and over every dtype pair, eager and
captured."""

from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu

if torch.cuda.is_available():
    from himuon_amd import _native as nat
    from himuon_amd.engine import AdamwTables, ApplyTables
    from himuon_amd.optimizers.himuon import HiMuon

DEV = "cuda"
F32, BF16 = torch.float32, torch.bfloat16
DTYPES = [torch.float32, torch.bfloat16, torch.float16]
BITS = {2: torch.int16, 4: torch.int32}
SCALE, ALPHA = [1 - 0.02 * 0.1, 1.0], [-0.02, -0.003]


@pytest.mark.parametrize("gdt", DTYPES)
@pytest.mark.parametrize("pdt", DTYPES)
def test_adamw_apply_equals_step_then_apply(gdt, pdt):
    gen = torch.Generator().manual_seed(2)
    sizes = [1, 7, 8, 4095, 4096, 4097, 20001]
    sa = torch.zeros(2 * nat.APPLY_MAX_GROUPS, device=DEV)
    nat.write_scale_alpha(sa, SCALE, ALPHA)
    sides = []
    data = [[torch.randn(n, generator=gen) * s for s in (1e-3, 1e-4, 1e-6, 0.02)] for n in sizes]
    for _ in range(2):
        entries, params = [], []
        for i, (g, m, v, p) in enumerate(data):
            g, m, v = (t.to(gdt).to(DEV) for t in (g, m, v.abs()))
            entries.append((g, m, v, torch.empty_like(g), torch.full((), float(i), device=DEV), i % 2))
            params.append(p.to(pdt).to(DEV))
        sides.append((entries, params))
    (e0, p0), (e1, p1) = sides
    b, eps = [0.95, 0.9], [1e-8, 1e-6]
    for _ in range(3):
        AdamwTables(e0).run(b, b, eps)
        ApplyTables([(p, e[3], e[5]) for p, e in zip(p0, e0)]).run(SCALE, ALPHA)
        fused = AdamwTables(e1, p1)
        assert all(fused.applied) and not fused.fallback
        fused.run(b, b, eps, sa)
    for a, c, p, q in zip(e0, e1, p0, p1):
        for k in (1, 2, 4):
            assert torch.equal(a[k], c[k])
        # (bits: fp16 second moments underflow to zero here, so some updates are infinite or NaN)
        assert torch.equal(p.view(BITS[p.element_size()]), q.view(BITS[q.element_size()]))


@pytest.mark.parametrize("cuda_graph", [False, True])
def test_optimizer_with_and_without(cuda_graph):
    gen = torch.Generator().manual_seed(3)
    vals = [torch.randn(*s, generator=gen) * 0.02 for s in ((999, 64), (64,), (256, 320), (33, 5))]
    runs = []
    for fuse in (True, False):
        ps = [torch.nn.Parameter(v.to(torch.bfloat16).to(DEV)) for v in vals]
        for p in ps:
            p.grad = torch.zeros_like(p)
        opt = HiMuon([{"params": [ps[2]], "use_muon": True},
                      {"params": [ps[0], ps[3]], "use_muon": False, "lr": 2e-3, "weight_decay": 0.1},
                      {"params": [ps[1]], "use_muon": False, "lr": 1e-3, "weight_decay": 0.0}],
                     lr=0.02, tile_size=128, cuda_graph=cuda_graph, cuda_graph_warmup=1)
        opt._fuse_adamw, opt._fuse_untile = fuse, True
        gg = torch.Generator().manual_seed(4)
        for k in range(5):
            for p in ps:
                p.grad.copy_((torch.randn(p.shape, generator=gg) * 1e-3).to(p.dtype))
            opt.param_groups[1]["lr"] = 2e-3 / (k + 1)
            opt.step()
        if fuse:
            assert not opt._adamw_updates
        runs.append(ps)
    # (eager, unfused: torch's own adds, the same arithmetic where the dtypes agree)
    for a, b in zip(*runs):
        assert torch.equal(a, b)


@pytest.mark.parametrize("cuda_graph", [False, True], ids=["eager", "captured"])
@pytest.mark.parametrize("gdt", DTYPES)
@pytest.mark.parametrize("pdt", DTYPES)
def test_optimizer_of_mixed_dtypes(pdt, gdt, cuda_graph):
    """Every pair of parameter and grad dtype, on norms, odd lengths, tails and a
    length that torch's vectorised add covers: the parameters of the step with
    and without the WD/LR inside it, which in an eager step is torch's own two
    ops on an update of the grad's dtype."""
    gen = torch.Generator().manual_seed(6)
    shapes = [(1,), (7,), (64,), (1000,), (33, 5), (4097,), (1 << 16,), (999, 64)]
    vals = [torch.randn(*s, generator=gen) * 0.02 for s in shapes]
    runs = []
    for fuse in (True, False):
        ps = [torch.nn.Parameter(v.to(pdt).to(DEV)) for v in vals]
        for p in ps:
            if pdt != gdt:
                p.grad_dtype = gdt
            p.grad = torch.zeros(p.shape, dtype=gdt, device=DEV)
        opt = HiMuon([{"params": ps[::2], "use_muon": False, "lr": 2e-2, "weight_decay": 0.1},
                      {"params": ps[1::2], "use_muon": False, "lr": 1e-2, "weight_decay": 0.0}],
                     lr=0.02, tile_size=128, cuda_graph=cuda_graph, cuda_graph_warmup=1)
        opt._fuse_adamw = fuse
        gg = torch.Generator().manual_seed(4)
        for _ in range(4):
            for p in ps:
                p.grad.copy_(torch.randn(p.shape, generator=gg).to(gdt))
            opt.step()
        fused = fuse and (cuda_graph or pdt == F32 or pdt == gdt == BF16)
        assert len(opt._adamw_updates) == (0 if fused else len(ps))
        runs.append(ps)
    for a, b in zip(*runs):
        assert torch.equal(a.view(BITS[a.element_size()]), b.view(BITS[b.element_size()])), tuple(a.shape)


@pytest.mark.parametrize("pdt,gdt", [(F32, F32), (BF16, BF16), (F32, BF16)])
def test_parameters_over_one_memory_are_updated_in_turn(pdt, gdt):
    """Weights tied by their data (two Parameters over one tensor, and one that
    overlaps it in part): each one's decay and update, in order, as torch's ops
    apply them; their neighbours stay in the fused pass."""
    n = 6000
    runs = []
    for fuse in (True, False):
        gen = torch.Generator().manual_seed(8)
        data = (torch.randn(3 * n, generator=gen) * 0.02).to(pdt).to(DEV)
        ps = [torch.nn.Parameter(d) for d in (data[:n], data[:n], data[n // 2: n // 2 + n], data[2 * n:])]
        for p in ps:
            if pdt != gdt:
                p.grad_dtype = gdt
            p.grad = torch.randn(n, generator=gen).to(gdt).to(DEV)
        opt = HiMuon([{"params": ps, "use_muon": False, "lr": 2e-2, "weight_decay": 0.1}], lr=0.02, tile_size=128,
                     cuda_graph=False)
        opt._fuse_adamw = fuse
        for _ in range(3):
            opt.step()
        assert [a for a in opt._adamw_tables.applied] == [False, False, False, fuse]
        runs.append(data)
    assert torch.equal(*runs)


def test_a_parameter_whose_layout_changes_between_steps():
    """The same memory with other strides (``p.data = p.data.t()``): the update is
    added element by element, as torch's ops do, not in the old layout."""
    runs = []
    for fuse in (True, False):
        gen = torch.Generator().manual_seed(9)
        p = torch.nn.Parameter((torch.randn(96, 96, generator=gen) * 0.02).to(DEV))
        p.grad = torch.randn(96, 96, generator=gen).to(DEV)
        opt = HiMuon([{"params": [p], "use_muon": False, "lr": 2e-2, "weight_decay": 0.1}], lr=0.02, tile_size=128,
                     cuda_graph=False)
        opt._fuse_adamw = fuse
        opt.step()
        p.data = p.data.t()
        opt.step()
        assert opt._adamw_tables.applied == [False]
        runs.append(p.data)
    assert torch.equal(*runs)


def test_adamw_apply_argument_errors():
    import ctypes

    one = (ctypes.c_double * 1)(0.95)
    lib = nat.load()
    assert lib.himuon_adamw_apply(8, 1, 4, 0, 1, one, one, one, 1, 8, None, None) == -22
    assert lib.himuon_adamw_apply(8, 1, 4, 0, 3, one, one, one, 1, 8, 16, None) == -22
    assert lib.himuon_adamw_apply(None, 1, 4, 0, 1, one, one, one, 1, 8, 16, None) == -22
    assert lib.himuon_adamw_apply(8, 1, 4, 0, 1, one, one, one, 33, 8, 16, None) == -22
