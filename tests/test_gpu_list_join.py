"""GPU: the join over larger binary states by lists per position (k_match_lists) against the oracle, event
by event, and against the general join (forwarding forced on, and four waves per state): states of 256
to 12,000 edges, lists of 1 to thousands of entries (ordered by a lane, a wave and the workgroup in the
emit pass), patterns of one to four edges with loops, repeated and unshared variables, small states with
more than 255 labels, a cap that stops a run midway, and a state past the LDS (general join)."""
import random

import numpy as np
import pytest

from hypergraphrewritingengine_amd.rules import Request, rule_from_lists
from oracle import pyoracle as po
from tests.parity import assert_exact

pytestmark = pytest.mark.gpu

REL = 0x1 | 0x2 | 0x4 | 0x100


def _state(m, n, seed):
    rnd = random.Random(seed)
    return [[rnd.randrange(n), rnd.randrange(n)] for _ in range(m)]


def _hubs(degrees):
    edges, nxt = [], len(degrees)
    for h, d in enumerate(degrees):
        for i in range(d):
            edges.append([h, nxt] if i % 3 else [nxt, h])
            nxt += 1
    random.Random(1).shuffle(edges)
    return edges


# pattern, state: chosen so that the matches stay in the hundreds or low thousands
CASES = {
    "edge": ([[0, 1]], _state(300, 200, 1)),
    "loop": ([[0, 0]], _state(700, 60, 2)),
    "path": ([[0, 1], [1, 2]], _state(400, 300, 3)),
    "fork": ([[0, 1], [0, 2]], _state(600, 600, 4)),
    "fork-hubs": ([[0, 1], [0, 2]], _hubs([15, 16, 17, 24, 25, 26, 30, 100])),
    "meet-hub": ([[0, 2], [1, 2]], _hubs([90, 110, 180])),
    "two-cycle": ([[0, 1], [1, 0]], _state(2000, 70, 5)),
    "parallel": ([[0, 1], [0, 1]], _state(1500, 100, 6)),
    "loop-and-edge": ([[0, 0], [0, 1]], _state(2500, 400, 7)),
    "triangle": ([[0, 1], [1, 2], [2, 0]], _state(3000, 600, 8)),
    "triangle-hub": ([[0, 1], [1, 2], [2, 0]], _hubs([1500]) + _state(600, 120, 9)),
    "four-cycle": ([[0, 1], [1, 2], [2, 3], [3, 0]], _state(700, 200, 10)),
    "star": ([[0, 1], [0, 2], [0, 3]], _state(500, 500, 11)),
    "unshared": ([[0, 0], [1, 1]], _state(800, 100, 12) + [[i, i] for i in range(20)]),
    "wide-labels": ([[0, 1], [1, 0]], [[i, i + 1] for i in range(200)] + [[i + 1, i] for i in range(0, 60, 3)] +
                    [[300 + i, 300 + i] for i in range(20)]),
    "12000": ([[0, 1], [1, 0]], _state(12000, 1300, 13)),
}


@pytest.mark.parametrize("name", list(CASES))
def test_events_equal_oracle(ctx, name):
    lhs, state = CASES[name]
    req = Request([rule_from_lists(lhs, [[0, lhs[0][1]]])], state, 1, flags=REL)
    o = po.evolve(req)
    assert o.counts["events"] > 0
    assert_exact(ctx.evolve(req), o, tr=True)


@pytest.mark.parametrize("name", ["path", "fork-hubs", "triangle", "loop"])
def test_two_steps_equal_the_general_join(ctx, name):
    lhs, state = CASES[name]
    reqs = [Request([rule_from_lists(lhs, [[0, lhs[0][1]]]), rule_from_lists([[0, 0], [0, 1]], [[1, 1]])], state[:k], 2,
                    state_cap=cap, flags=REL) for k in (257, 300) for cap in (40, 20000)]
    want = [po.evolve(r) for r in reqs]
    for r, o in zip(ctx.evolve_batch(reqs), want):
        assert_exact(r, o, tr=True)
    try:
        ctx.set_forwarding(1)
        for r, o in zip(ctx.evolve_batch(reqs), want):
            assert np.array_equal(r.events(), o.events)
        ctx.set_forwarding(-1)
        ctx.set_join_team(4)
        for r, o in zip(ctx.evolve_batch(reqs), want):
            assert np.array_equal(r.events(), o.events)
    finally:
        ctx.set_forwarding(-1)
        ctx.set_join_team(0)


def test_state_past_the_lds(ctx):
    state = _state(21000, 15000, 14)
    req = Request([rule_from_lists([[0, 1], [1, 2], [2, 0]], [[0, 2], [2, 1], [1, 0]])], state, 1, flags=REL)
    assert_exact(ctx.evolve(req), po.evolve(req), tr=True)
