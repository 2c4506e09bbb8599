"""newton_schulz without copies: the one-launch form (himuon_ns_direct) and the
replayed launches that read the input and write the result in place
(himuon_write_desc) give the bits of the gather, normaliser, NS and untile
launches on a copy, for every dtype, at the edges of both ranges, from inputs
at any alignment and stride, and recorded into a caller's graph."""

from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu

if torch.cuda.is_available():
    from himuon_amd import _native as nat
    from himuon_amd import engine as E
    from himuon_amd.engine import newton_schulz

DEV = "cuda"
F32, BF16, F16 = torch.float32, torch.bfloat16, torch.float16
DIRECT = [(3, 128, 128), (2, 65, 65), (5, 100, 101), (1, 66, 128), (4, 129, 131), (2, 256, 256), (300, 200, 255), (96, 100),
          (256, 251)]
PLANNED = [(2, 64, 128), (3, 128, 129), (2, 256, 257), (2, 255, 130), (4, 384, 200), (130, 700)]


def _launches(G, steps):
    M, N = G.shape[-2:]
    plan = E._NsPlan(G.numel() // (M * N), M, N, G.dtype, G.device, G.ndim == 2, "auto")
    plan.xin.view(G.shape).copy_(G)
    plan._launches(steps)
    return plan.out.view(G.shape)


def _input(shape, dtype, seed):
    return (torch.randn(*shape, generator=torch.Generator().manual_seed(seed)) * 1e-3).to(dtype).to(DEV)


@pytest.mark.parametrize("shape", DIRECT + PLANNED, ids=lambda s: "x".join(map(str, s)))
@pytest.mark.parametrize("dtype", [F32, BF16, F16])
def test_equals_the_launches_on_a_copy(shape, dtype):
    M, N = shape[-2:]
    assert nat.ns_direct_supported(M, N, dtype) == (shape in DIRECT and M <= N)
    for k, steps in enumerate((5, 0, 1)):
        G = _input(shape, dtype, k)
        keep = G.clone()
        out = newton_schulz(G, steps=steps)
        assert torch.equal(G, keep) and out.dtype == dtype and out.is_contiguous()
        assert torch.equal(out, _launches(G, steps))


@pytest.mark.parametrize("shape", [(3, 100, 120), (3, 200, 300)])
def test_input_layouts(shape):
    G = _input(shape, F32, 7)
    ref = newton_schulz(G)
    buf = torch.zeros(G.numel() + 1, device=DEV)
    off = buf[1:].view(shape)  # contiguous, one element into its storage
    off.copy_(G)
    wide = torch.zeros(shape[0], shape[1], shape[2] + 5, device=DEV)
    wide[:, :, 2:-3] = G
    for x in (off, wide[:, :, 2:-3], G.transpose(1, 2).contiguous().transpose(1, 2), G.flip(0).flip(0)):
        assert torch.equal(newton_schulz(x), ref)
    d = newton_schulz(G.double())
    assert d.dtype == torch.float64 and torch.equal(d, ref.double())
    neg = torch._neg_view(-G)  # contiguous, its memory holds -G
    assert neg.is_neg() and neg.is_contiguous() and torch.equal(newton_schulz(neg), ref)
    p = G.clone().requires_grad_()
    assert torch.equal(newton_schulz(p), ref)
    nan = G.clone()
    nan[1, 3, 4] = float("nan")
    out = newton_schulz(nan)
    assert out[1].isnan().all() and torch.equal(out[0], ref[0]) and torch.equal(out[2], ref[2])


@pytest.mark.parametrize("shape", [(3, 100, 120), (2, 200, 300)])
def test_in_a_callers_graph(shape):
    a, b = _input(shape, F32, 8), _input(shape, F32, 9)
    ref = [newton_schulz(a), newton_schulz(b)]
    static = a.clone()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = newton_schulz(static)
    for k in (0, 1, 0):
        static.copy_((a, b)[k])
        graph.replay()
        other = newton_schulz((b, a)[k])  # eager work between the replays
        torch.cuda.synchronize()
        assert torch.equal(out, ref[k]) and torch.equal(other, ref[1 - k])


def test_refuses_other_shapes():
    lib = nat.load()
    args = [8, 16, 0, 128, 128, 0, 5, 1.0, 1.0, 1.0, 1e-7, 0x10, None]
    assert lib.himuon_ns_direct(*args) == 0  # empty work: no launch
    for pos, val in [(3, 64), (3, 129), (4, 257), (4, 127), (5, 3), (6, -1), (11, 1), (0, None), (1, None), (2, -1), (2, 1 << 31)]:
        bad = list(args)
        bad[pos] = val
        assert lib.himuon_ns_direct(*bad) == -22, (pos, val)
    assert lib.himuon_write_desc(None, 8, None) == -22
