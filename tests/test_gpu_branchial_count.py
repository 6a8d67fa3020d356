"""GPU: the branchial pair counts of rules of at most three LHS edges (k_branchial_count) against the
oracle's: parents of 1 to 130 edges (the last by lists), rules of one, two and three edges alone and
mixed, every order of an edge pair and triple matched, parents with hundreds of matches and with more than
1,024 (a wave each), and more than 16,384 parents (16 lanes each, the larger ones by bit sets),
a rule of four edges beside them (bit sets), and per-parent counts behind the recorded pairs."""
import random

import pytest

from hypergraphrewritingengine_amd.rules import Request, rule_from_lists
from oracle import pyoracle as po
from tests.parity import assert_exact

pytestmark = pytest.mark.gpu

REL = 0x1 | 0x2 | 0x4 | 0x100
RULES = {
    "one": [rule_from_lists([[0, 1]], [[0, 1], [1, 2]])],
    "two": [rule_from_lists([[0, 1], [0, 2]], [[0, 1]])],
    "both-orders": [rule_from_lists([[0, 1], [1, 0]], [[0, 1]]), rule_from_lists([[0, 1], [2, 1]], [[0, 2]])],
    "mixed": [rule_from_lists([[0, 0]], [[0, 1]]), rule_from_lists([[0, 1], [1, 2]], [[0, 2]])],
    "triangles": [rule_from_lists([[0, 1], [1, 2], [2, 0]], [[0, 1]]), rule_from_lists([[0, 1], [2, 1], [2, 0]], [[0, 2]])],
    "four": [rule_from_lists([[0, 1], [1, 2], [2, 3], [3, 0]], [[0, 1]])],
    "three": [rule_from_lists([[0, 1], [1, 2], [2, 3]], [[0, 3]]), rule_from_lists([[0, 1], [0, 2]], [[1, 2]])],
}


def _state(m, seed):
    rnd = random.Random(seed)
    n = max(1, m // 2 if m < 40 else m)
    return [[rnd.randrange(n), rnd.randrange(n)] for _ in range(m)]


@pytest.mark.parametrize("name", list(RULES))
def test_pairs_equal_oracle(ctx, name):
    for m in (1, 2, 3, 15, 16, 17, 31, 33, 63, 64, 65, 127, 128, 129, 130):
        req = Request(RULES[name], _state(m, m), 1, flags=REL)
        assert_exact(ctx.evolve(req), po.evolve(req), tr=True)
    dense = Request(RULES[name], [[i, j] for i in range(5) for j in range(5)] * 2, 1, flags=REL)
    if name != "four":                                       # (11 million pairs)
        assert_exact(ctx.evolve(dense), po.evolve(dense), tr=True)
    star = Request(RULES[name], [[0, i % 20] for i in range(24)], 2, state_cap=700, flags=REL)
    assert_exact(ctx.evolve(star), po.evolve(star), tr=True)


@pytest.mark.parametrize("flags", [REL, 0x3])
def test_many_parents(ctx, flags):
    reqs = [Request(RULES[("mixed", "two", "three", "four")[i % 4]], _state(1 + i * 5 % 128, i), 1, flags=flags) for i in range(120)]
    want = [po.evolve(r) for r in reqs]
    got = ctx.evolve_batch([reqs[i % 120] for i in range(16500)])
    for i in list(range(0, 120)) + [16384 + k for k in range(116)]:
        if flags == REL and i < 120:
            assert_exact(got[i], want[i % 120], tr=True)
        assert got[i].counts["branchial_pairs"] == len(want[i % 120].branchial), i
