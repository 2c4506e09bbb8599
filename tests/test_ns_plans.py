"""Which device state newton_schulz calls share: the ones of one stream and
shape, and nothing else; the kept plans are bounded."""

from __future__ import annotations

import pytest
import torch

from himuon_amd import engine as E


@pytest.fixture
def plans(monkeypatch):
    kept: dict = {}
    monkeypatch.setattr(E, "_NS_PLANS", kept)
    monkeypatch.setattr(E, "_NsPlan", lambda *spec: [spec])  # (a new object each)
    return kept


def test_streams_share_no_plan(plans):
    a, b = E._ns_plan(7, 3, 512, 512), E._ns_plan(8, 3, 512, 512)
    assert a is not b
    assert E._ns_plan(7, 3, 512, 512) is a and E._ns_plan(8, 3, 512, 512) is b
    assert E._ns_plan(7, 3, 512, 640) is not a


def test_the_least_recently_used_plans_make_room(plans):
    first = [E._ns_plan(0, k) for k in range(E._NS_PLANS_MAX)]
    other = E._ns_plan(1, 0)
    assert E._ns_plan(0, 0) is first[0]
    E._ns_plan(0, 99)  # drops shape 1 of stream 0, and nothing of stream 1
    assert E._ns_plan(0, 0) is first[0] and E._ns_plan(1, 0) is other
    assert E._ns_plan(0, 1) is not first[1]
    for s in range(3 * E._NS_PLANS_TOTAL):
        E._ns_plan(s, s)
        assert len(plans) <= E._NS_PLANS_TOTAL
        assert sum(k[0] == 0 for k in plans) <= E._NS_PLANS_MAX


def test_an_unknown_family_is_refused_and_not_kept(monkeypatch):
    kept: dict = {}
    monkeypatch.setattr(E, "_NS_PLANS", kept)
    with pytest.raises(ValueError):
        E._ns_plan(0, 2, 300, 300, torch.float32, torch.device("cpu"), False, "fastest")
    assert not kept


def test_what_is_launched_unrecorded():
    """The shapes whose iterations are one launch, as bench.ns_family names their kernels."""
    from bench import ns_family
    from himuon_amd import _native as nat

    for M in (1, 16, 17, 32, 33, 64, 65, 128, 129, 256, 257, 512):
        for N in (16, 128, 129, 256, 257, 384, 512, 513, 768, 1024, 1280, 1536, 2048, 2300):
            m, _, mp, np_, _ = nat.ns_geometry(M, N)
            for family in nat.NS_FAMILIES:
                one = family == "auto" and ns_family(mp, np_, family, m) in ("few_rows", "lds")
                assert nat.one_launch(m, mp, np_, family) == one, (M, N, family)
