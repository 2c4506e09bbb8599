"""Which device state newton_schulz calls share: the ones of one stream and
shape, and nothing else; the kept plans are bounded."""

from __future__ import annotations

import pytest

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
