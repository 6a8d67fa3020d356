"""GPU: the join by bit sets (small binary states) against the oracle, event by event, and against the
list join (forced by four waves per state): states of 63 to 256 edges (one, two and four words per
set, and one edge past them), the vertex-label limit and one past it, patterns of one to four edges
with loops, repeated and unshared variables, a pattern edge that is not binary, more than two rules,
a five-edge pattern (list join), every lane count, and caps that stop a run midway."""
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


PATTERNS = {
    "edge": [[0, 1]],
    "loop": [[0, 0]],
    "path": [[0, 1], [1, 2]],
    "fork": [[0, 1], [0, 2]],
    "meet": [[0, 2], [1, 2]],
    "two-cycle": [[0, 1], [1, 0]],
    "parallel": [[0, 1], [0, 1]],
    "loop-and-edge": [[0, 0], [0, 1]],
    "triangle": [[0, 1], [1, 2], [2, 0]],
    "reversed-order": [[1, 2], [0, 1], [2, 2]],
    "four-cycle": [[0, 1], [1, 2], [2, 3], [3, 0]],
    "star": [[0, 1], [0, 2], [0, 3]],
    "five": [[0, 1], [1, 2], [2, 3], [3, 4], [4, 0]],
    "ternary-edge": [[0, 1], [1, 2, 0]],
}


@pytest.mark.parametrize("name", list(PATTERNS))
def test_patterns_equal_oracle(ctx, name):
    rule = rule_from_lists(PATTERNS[name], [[0, 1], [1, 5]])
    reqs = [Request([rule], _state(m, n, m), 2, flags=REL, state_cap=1500)
            for m, n in ((1, 2), (9, 3), (20, 40), (63, 60), (64, 70), (65, 60), (100, 120))]
    want = [po.evolve(r) for r in reqs]
    try:
        for lanes in (0, 16, 32, 64):
            ctx.set_join_lanes(lanes)
            for r, o in zip(ctx.evolve_batch(reqs), want):
                assert_exact(r, o, tr=True)
        ctx.set_join_lanes(0)
        ctx.set_join_team(4)
        for r, o in zip(ctx.evolve_batch(reqs), want):
            assert np.array_equal(r.events(), o.events) and np.array_equal(r.states()[0], o.state_hash)
    finally:
        ctx.set_join_lanes(0)
        ctx.set_join_team(0)


def test_unshared_variables(ctx):
    rule = rule_from_lists([[0, 1], [2, 3]], [[0, 3]])
    req = Request([rule], _state(12, 8, 3), 2, flags=REL)
    assert_exact(ctx.evolve(req), po.evolve(req), tr=True)


@pytest.mark.parametrize("m,n", [(127, 100), (128, 100), (129, 100), (253, 200), (254, 253), (255, 254), (256, 255),
                                 (250, 256)])
def test_sizes_equal_oracle(ctx, m, n):
    edges = [[i % n, (i * 5 + 1) % n] for i in range(n)] + _state(m - n, n, m) if m > n else \
            [[i, (i * 7 + 1) % n] for i in range(m)] + [[n - 1, n - 2]]
    for rule in (rule_from_lists([[0, 1], [1, 2]], [[0, 2]]), rule_from_lists([[0, 1], [1, 0]], [[0, 0], [1, 1]])):
        req = Request([rule], edges, 1, flags=REL)
        assert_exact(ctx.evolve(req), po.evolve(req), tr=True)


def test_many_rules_and_caps(ctx):
    rules = [rule_from_lists(PATTERNS[k], [[0, 1], [0, 5]]) for k in ("edge", "fork", "triangle", "loop")]
    reqs = [Request(rules[:k], _state(10 + 7 * i, 12, i), 3, flags=REL, state_cap=cap)
            for i in range(6) for k in (1, 2, 4) for cap in (50, 700)]
    for r, req in zip(ctx.evolve_batch(reqs), reqs):
        assert_exact(r, po.evolve(req), tr=True)
