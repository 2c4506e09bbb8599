"""Which tensors of a list share memory, against comparing every pair."""

from __future__ import annotations

import random

import torch

from himuon_amd.engine import mem_span, sharing


def test_against_every_pair():
    rng = random.Random(5)
    buf = torch.zeros(200)
    for _ in range(300):
        ts = []
        for _ in range(rng.randint(0, 7)):
            a = rng.randint(0, 190)
            ts.append(buf[a: a + rng.choice((0, 1, 3, 10, 60)) : rng.choice((1, 1, 2))])
        want = set()
        for i, s in enumerate(map(mem_span, ts)):
            for j, t in enumerate(map(mem_span, ts)):
                if i != j and max(s[0], t[0]) < min(s[1], t[1]):
                    want |= {i, j}
        assert sharing(ts) == want


def test_spans():
    b = torch.zeros(4, 6)
    p = b.data_ptr()
    assert mem_span(b) == (p, p + 96) and mem_span(b[1:3, 2:4]) == (p + 32, p + 64)
    assert mem_span(b.t()) == (p, p + 96) and mem_span(b[:, :1].expand(4, 6)) == (p, p + 76)
    assert mem_span(torch.zeros(0, 3)) == (0, 0)
