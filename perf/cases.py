"""The work that a program using this framework has it do, as measurable cases.

Three kinds of case:

* ``step``: one ``optimizer.step()`` of the HiMuon optimizer built by
  ``get_optimizer("himuon", model, args)``: momentum, tiling, Newton-Schulz per
  tile (or per matrix), the update with weight decay and learning rate, and
  the AdamW groups (embedding, norms) where the model has them. What comes back
  is the updated parameters, momentum buffers and AdamW moments.
* ``ns``: one ``HiMuon.newton_schulz(G)`` call on a batch or a single matrix.
* ``products``: one Newton-Schulz iteration through the kernel API
  (``XXT``, ``ba_plus_cAA``, ``fused_bmm_add``) in the operand dtype of the case.

The matrices of one shape live in one stacked buffer (each matrix in an
aligned slot of its own), as a program with flat parameter storage keeps them;
the outputs are those buffers.
"""

from __future__ import annotations

import math

import torch

from himuon_amd import kernels as K
from himuon_amd.optim import get_optimizer
from himuon_amd.optimizers.himuon import HiMuon

NS_A, NS_B, NS_C = 3.4445, -4.7750, 2.0315
FULL = 1_000_000_000  # tile_size of the full-matrix (Muon) mode
LR, WD, MU, ADAMW_LR, BETA, EPS = 0.02, 0.1, 0.95, 0.02, 0.95, 1e-8
ADAMW_STEPS = 100  # AdamW steps taken before the measured one
SLOT = 256  # elements: every matrix starts on a multiple of this in its buffer
DTYPES = {"fp32": torch.float32, "bf16": torch.bfloat16, "fp16": torch.float16}

QWEN_06B = "2048x1024 1024x1024 1024x1024 1024x2048 3072x1024 3072x1024 1024x3072"
QWEN_4B = "4096x2560 1024x2560 1024x2560 2560x4096 9728x2560 9728x2560 2560x9728"
LLAMA_8B = "4096x4096 1024x4096 1024x4096 4096x4096 14336x4096 14336x4096 4096x14336"


def _step(name, layers, shapes, tile, tile_w=None, param="bf16", grad="fp32", embed=0, graph=True):
    return {"name": name, "kind": "step", "layers": layers, "shapes": shapes, "tile_h": tile, "tile_w": tile_w or tile,
            "param": param, "grad": grad, "embed": embed, "graph": graph}


def listed():
    return [
        # the smallest step: one weight matrix, where launches and latency are all there is
        _step("step_one_matrix_t256", 1, "1024x1024", 256, param="fp32"),
        # a small stack of linear layers in pure bf16 (the optimizer-step micro-benchmark's shape)
        _step("step_8_linear_t512", 8, "2048x2048", 512, grad="bf16"),
        # a whole small language model at the default tile: hidden matrices on Muon, embedding and norms on AdamW
        _step("step_0.6b_t512_adamw", 28, QWEN_06B, 512, embed=151936),
        # the same hidden matrices at a smaller tile
        _step("step_0.6b_t256", 28, QWEN_06B, 256),
        # the same hidden matrices in full-matrix mode (plain Muon)
        _step("step_0.6b_full", 28, QWEN_06B, FULL),
        # the largest: the headline workload, all hidden matrices of a 4B model at the default tile
        _step("step_4b_t512", 36, QWEN_4B, 512),
        # very many small tiles, all in fp32: a quarter of an 8B model's layers at tile 128
        _step("step_8b_quarter_t128", 8, LLAMA_8B, 128, param="fp32"),
        # sizes that are no multiples of anything, full-matrix mode, pure bf16
        _step("step_ragged_full", 12, "880x880 220x880 880x880 2345x880 880x2345", FULL, grad="bf16"),
        # ragged tiles without graph capture: a program whose steps run eagerly
        _step("step_ragged_eager_t512", 16, "1000x1000 2730x1000 1000x2730", 512, graph=False),
        # the Newton-Schulz call alone, many small tiles (the kernel micro-benchmark's shape)
        {"name": "ns_512x128x128", "kind": "ns", "batch": 512, "m": 128, "n": 128, "dtype": "bf16"},
        # the Newton-Schulz call on one weight's momentum, as a hand-written Muon loop makes it
        {"name": "ns_3072x1024", "kind": "ns", "batch": 0, "m": 3072, "n": 1024, "dtype": "fp32"},
        # one iteration through the kernel API in fp32, for studies of the iteration's precision
        {"name": "products_8x512x1024_fp32", "kind": "products", "batch": 8, "m": 512, "n": 1024, "dtype": "fp32"},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _size(rng, lo, hi):
    """A size of lo .. hi, log-uniform: half of them as drawn, the others rounded to a multiple of 64 or 128."""
    v = _log(rng, lo, hi)
    r = rng.choice((1, 1, 64, 128))
    return max(lo, v // r * r)


def draw(rng):
    kind = rng.choice(("step",) * 6 + ("ns", "ns", "products"))
    if kind == "ns":
        m, n = _size(rng, 64, 2048), _size(rng, 64, 3072)
        most = max(1, (1 << 26) // (m * n))
        return {"kind": "ns", "batch": rng.choice((0, _log(rng, 1, min(2048, most)))), "m": m, "n": n,
                "dtype": rng.choice(("bf16", "fp32"))}
    if kind == "products":
        m, n = _size(rng, 64, 1024), _size(rng, 64, 2048)
        return {"kind": "products", "batch": _log(rng, 1, 64), "m": m, "n": n,
                "dtype": rng.choice(("bf16", "fp16", "fp32"))}
    hidden = _size(rng, 256, 4096)
    ffn = _size(rng, 2 * hidden, 4 * hidden)
    kv = max(64, hidden // rng.choice((1, 2, 4)))
    shapes = "%dx%d %dx%d %dx%d %dx%d %dx%d" % (hidden, hidden, kv, hidden, hidden, hidden, ffn, hidden, hidden, ffn)
    per_layer = sum(h * w for h, w in _shapes(shapes))
    tile = rng.choice(((512, 512), (512, 512), (256, 256), (128, 128), (1024, 1024), (384, 384), (256, 512), (FULL, FULL)))
    # at most 1.5 G elements, or 0.15 G where whole matrices are iterated
    layers = _log(rng, 1, max(1, min(32, (150_000_000 if tile[0] == FULL else 1_500_000_000) // per_layer)))
    param, grad = rng.choice((("bf16", "fp32"), ("bf16", "fp32"), ("bf16", "bf16"), ("fp32", "fp32")))
    return {"kind": "step", "layers": layers, "shapes": shapes, "tile_h": tile[0], "tile_w": tile[1], "param": param,
            "grad": grad, "embed": rng.choice((0, 0, _log(rng, 1000, 150_000))), "graph": rng.random() < 0.8}


# -- inputs ---------------------------------------------------------------------


def _shapes(text):
    return [tuple(int(v) for v in s.split("x")) for s in text.split()]


def _generator(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _stacks(case):
    """(count, h, w or 0) of every stacked buffer: the hidden matrices by
    shape position, then the embedding and the norms (1-D, w = 0)."""
    shapes = _shapes(case["shapes"])
    out = [(case["layers"], h, w) for h, w in shapes]
    if case["embed"]:
        out += [(1, case["embed"], shapes[0][1]), (2 * case["layers"] + 1, shapes[0][1], 0)]
    return out


def _fill(case, seed, bufs=None):
    """The step's inputs, per stack: parameters, grads and optimizer state
    (momentum, or the two AdamW moments) as they are in the middle of training."""
    gen = _generator(seed)
    pdt, gdt = DTYPES[case["param"]], DTYPES[case["grad"]]
    stacks = _stacks(case)
    muon = len(_shapes(case["shapes"]))
    if bufs is None:
        bufs = []
        for i, (count, h, w) in enumerate(stacks):
            size = (count, -(-h * max(w, 1) // SLOT) * SLOT)
            bufs.append([torch.empty(size, device="cuda", dtype=dt) for dt in (pdt, gdt, gdt) + (gdt,) * (i >= muon)])
    for i, b in enumerate(bufs):
        b[0].normal_(0.0, 0.02, generator=gen)
        b[1].normal_(0.0, 1e-3, generator=gen)
        if i < muon:  # momentum 0.95 of such grads
            b[2].normal_(0.0, 3.2e-3, generator=gen)
        else:
            b[2].normal_(0.0, 1.6e-4, generator=gen)
            b[3].normal_(1e-6, 1e-7, generator=gen).abs_()
    return bufs


def _views(buf, count, h, w):
    """The matrices (or vectors) of a stacked buffer."""
    n = h * max(w, 1)
    return [buf[i, :n].view(h, w) if w else buf[i, :n] for i in range(count)]


def prepare(case, seed):
    if case["kind"] == "ns":
        shape = (case["batch"],) * (case["batch"] > 0) + (case["m"], case["n"])
        G = torch.empty(shape, device="cuda", dtype=DTYPES[case["dtype"]]).normal_(0.0, 1e-3, generator=_generator(seed))
        return {"case": case, "G": G}
    if case["kind"] == "products":
        X, A, B = _products_inputs(case, seed)
        return {"case": case, "X": X, "A": A, "B": B}
    bufs = _fill(case, seed)
    net = torch.nn.Module()
    for i, ((count, h, w), b) in enumerate(zip(_stacks(case), bufs)):
        for j, (p, g) in enumerate(zip(_views(b[0], count, h, w), _views(b[1], count, h, w))):
            p = torch.nn.Parameter(p)
            if p.dtype != g.dtype:
                p.grad_dtype = g.dtype
            p.grad = g
            adamw2d = case["embed"] and i == len(bufs) - 2
            net.register_parameter("embed_tokens" if adamw2d else "layer%d_w%d" % (j, i), p)
    args = {"lr": LR, "weight_decay": WD, "momentum": MU, "tile_size": (case["tile_h"], case["tile_w"]),
            "cuda_graph": case["graph"]}
    opt = get_optimizer("himuon", net, args)
    for group in opt.param_groups:
        if not group["use_muon"]:
            group["lr"] = ADAMW_LR
    # the optimizer state, in stacked buffers too
    params, steps = list(net.parameters()), []
    for i, ((count, h, w), b) in enumerate(zip(_stacks(case), bufs)):
        for j in range(count):
            st = opt.state[params.pop(0)]
            if len(b) == 3:
                st["momentum_buffer"] = _views(b[2], count, h, w)[j]
            else:
                st["step"] = torch.zeros((), device="cuda")
                st["moment1"], st["moment2"] = _views(b[2], count, h, w)[j], _views(b[3], count, h, w)[j]
                steps.append(st["step"])
    # the plan, the device buffers and the captured step that a program has after its first steps
    for _ in range(4 if case["graph"] else 1):
        opt.step()
    _fill(case, seed, bufs)
    for s in steps:
        s.fill_(ADAMW_STEPS)
    return {"case": case, "opt": opt, "net": net, "out": [[b[0]] + b[2:] for b in bufs]}


def _products_inputs(case, seed):
    b, m, n = case["batch"], case["m"], case["n"]
    dt = DTYPES[case["dtype"]]
    X = torch.empty((b, m, n), device="cuda", dtype=torch.float32).normal_(0.0, 1.0, generator=_generator(seed))
    X = (X / math.sqrt(m * n)).to(dt)
    return X, torch.empty((b, m, m), device="cuda", dtype=dt), torch.empty((b, m, m), device="cuda", dtype=dt)


def run(state):
    kind = state["case"]["kind"]
    if kind == "ns":
        return HiMuon.newton_schulz(state["G"])
    if kind == "products":
        X, A, B = state["X"], state["A"], state["B"]
        K.XXT(X, A)
        K.ba_plus_cAA(A, NS_C, NS_B, B)
        return A, B, K.fused_bmm_add(B, X, NS_A)
    state["opt"].step()
    return state["out"]


# -- what a pass cannot do without ----------------------------------------------


def _blocks(case, h, w):
    """(count, rows, columns) of the matrices NS runs on, of one h x w parameter."""
    th, tw = case["tile_h"], case["tile_w"]
    if h * w <= th * tw:
        return [(1, h, w)]
    rows = [(h // th, th), (1, h % th)]
    cols = [(w // tw, tw), (1, w % tw)]
    return [(a * b, r, c) for a, r in rows for b, c in cols if a * b and r and c]


def _ns_flops(m, n):
    """Five iterations on m x n: B X whole, half of each of the two symmetric products."""
    m, n = min(m, n), max(m, n)
    return 5.0 * (m * m * n + m**3 + 2 * m * m * n)


def work(case):
    if case["kind"] == "ns":
        b, m, n = max(1, case["batch"]), case["m"], case["n"]
        return {"bytes": 2 * b * m * n * DTYPES[case["dtype"]].itemsize, "flops": b * _ns_flops(m, n)}
    if case["kind"] == "products":
        b, m, n = case["batch"], case["m"], case["n"]
        # each call reads its operands and writes its result
        moved = (m * n + m * m) + 2 * m * m + (m * m + 2 * m * n)
        return {"bytes": b * moved * DTYPES[case["dtype"]].itemsize, "flops": b * (m * m * n + m**3 + 2.0 * m * m * n)}
    ps, gs = DTYPES[case["param"]].itemsize, DTYPES[case["grad"]].itemsize
    muon = len(_shapes(case["shapes"]))
    moved = flops = 0.0
    for i, (count, h, w) in enumerate(_stacks(case)):
        n = count * h * max(w, 1)
        moved += n * (2 * ps + gs + (2 if i < muon else 4) * gs)
        if i < muon:
            flops += sum(count * c * _ns_flops(r, s) for c, r, s in _blocks(case, h, w))
    return {"bytes": moved, "flops": flops}


# -- the same in 64 bits ---------------------------------------------------------


def _ns64(X):
    """Newton-Schulz of a float64 batch (B, m, n)."""
    if X.shape[1] > X.shape[2]:
        return _ns64(X.transpose(1, 2).contiguous()).transpose(1, 2)
    X = X / (X.square().sum(dim=(1, 2), keepdim=True).sqrt() + 1e-7)
    for _ in range(5):
        A = torch.bmm(X, X.transpose(1, 2).contiguous())
        B = NS_B * A + NS_C * torch.bmm(A, A)
        X = NS_A * X + torch.bmm(B, X)
    return X


def _update64(E, case):
    """The lr-adjusted update of one float64 momentum matrix."""
    h, w = E.shape
    th, tw = case["tile_h"], case["tile_w"]
    if h * w <= th * tw:
        return _ns64(E[None])[0] * (0.2 * math.sqrt(max(h, w)))
    R, C = -(-h // th), -(-w // tw)
    T = torch.nn.functional.pad(E, (0, C * tw - w, 0, R * th - h))
    T = T.view(R, th, C, tw).permute(0, 2, 1, 3).reshape(R * C, th, tw)
    U = torch.cat([_ns64(t) for t in T.split(max(1, (1 << 28) // (th * tw)))])
    U = U.view(R, C, th, tw).permute(0, 2, 1, 3).reshape(R * th, C * tw)[:h, :w]
    return U * (0.2 * math.sqrt(max(th, tw)))


def exact(case, seed):
    if case["kind"] == "ns":
        G = prepare(case, seed)["G"].double()
        return _ns64(G[None])[0] if G.ndim == 2 else _ns64(G)
    if case["kind"] == "products":
        X = _products_inputs(case, seed)[0].double()
        A = torch.bmm(X, X.transpose(1, 2).contiguous())
        B = NS_C * torch.bmm(A, A) + NS_B * A
        return A, B, torch.bmm(B, X) + NS_A * X
    muon = len(_shapes(case["shapes"]))
    out = []
    for i, ((count, h, w), b) in enumerate(zip(_stacks(case), _fill(case, seed))):
        if i < muon:
            p, m = b[0].double(), b[2].double()
            for pv, g, mv in zip(_views(p, count, h, w), _views(b[1], count, h, w), _views(m, count, h, w)):
                mv.mul_(MU).add_(g.double())
                pv.mul_(1 - LR * WD).sub_(LR * _update64(g.double() + MU * mv, case))
            out.append([p, m])
        else:
            n = h * max(w, 1)
            p, g, m, v = (t.double() for t in b)
            pv, gv, mv, vv = p[:, :n], g[:, :n], m[:, :n], v[:, :n]
            mv.mul_(BETA).add_(gv, alpha=1 - BETA)
            vv.mul_(BETA).addcmul_(gv, gv, value=1 - BETA)
            bc = 1 - BETA ** (ADAMW_STEPS + 1)
            u = (mv / bc) / ((vv / bc).sqrt() + EPS)
            pv.mul_(1 - ADAMW_LR * (WD if w else 0.0)).sub_(ADAMW_LR * u)
            out.append([p, m, v])
    return out


def tolerance(case):
    """About four times what one correct evaluation was measured to be off the
    float64 one. Newton-Schulz in bf16 amplifies the rounding of the small
    singular values: 0.9 to 1.4 % of the result (two summation orders differ by
    as much); in the parameters that is 0.25 %, with bf16 parameters' own
    rounding 0.36 %. The products: 0.0022 in bf16, an eighth of that in fp16
    (three more bits), 3.4e-6 in fp32 (16 significant bits of each operand)."""
    if case["kind"] == "ns":
        return {"rel": 5e-2}
    if case["kind"] == "products":
        return {"rel": {"bf16": 9e-3, "fp16": 1.2e-3, "fp32": 1.5e-5}[case["dtype"]]}
    return {"rel": 1.4e-2 if case["param"] == "bf16" else 1e-2}
