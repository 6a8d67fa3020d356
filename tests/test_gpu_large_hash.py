"""GPU: states of one arity hashed with their colours in LDS (k_wl_large, k_expand_large) against the
oracle, and the expansion against the general one (two waves per child): neighbour lists of 8, 9, 16,
17, 64, 65 and thousands of entries, a list longer than the labels (parallel edges), arities 2 to 4,
many components and one, sizes on both sides of the layouts (everything in LDS or not) and of the limits
on labels and list entries, a few states and more than the chip holds at once."""
import random

import numpy as np
import pytest

from hypergraphrewritingengine_amd.rules import Request, rule_from_lists
from oracle import pyoracle as po
from tests.parity import assert_exact

pytestmark = pytest.mark.gpu

REL = 0x1 | 0x2 | 0x4 | 0x100


def _state(m, n, a, seed):
    rnd = random.Random(seed)
    return [[rnd.randrange(n) for _ in range(a)] for _ in range(m)]


def _dense(edges):
    ids = {}
    return [[ids.setdefault(v, len(ids)) for v in e] for e in edges]


def _hubs(m, degrees):
    """m edges: hubs of the given degrees on leaves, then a path."""
    edges, nxt = [], len(degrees)
    for h, d in enumerate(degrees):
        for i in range(d):
            edges.append([h, nxt] if i % 2 else [nxt, h])
            nxt += 1
    while len(edges) < m:
        edges.append([nxt, nxt + 1])
        nxt += 1
    return edges


STATES = {
    "hubs": lambda: _hubs(900, [8, 9, 15, 16, 17, 31, 32, 33, 63, 64, 65, 66, 128, 200]),
    "star": lambda: _hubs(2000, [2000]),
    "two-stars": lambda: _hubs(6000, [2500, 2500]),
    "parallel": lambda: [[0, 1]] * 1500 + [[1, 2]] * 700,
    "loops": lambda: [[0, 0]] * 1200,
    "sparse-3000": lambda: _state(3000, 3000, 2, 1),
    "sparse-7001": lambda: _state(7001, 8000, 2, 2),
    "sparse-12000": lambda: _state(12000, 12300, 2, 3),
    "labels-16383": lambda: [[i, i + 1] for i in range(16382)],
    "labels-16384": lambda: [[i, i + 1] for i in range(16383)],
    "dense-30": lambda: _state(1200, 30, 2, 4),
    "ternary-900": lambda: _state(900, 500, 3, 5),
    "ternary-10922": lambda: _state(10922, 6000, 3, 6),
    "ternary-10923": lambda: _state(10923, 6000, 3, 6),
    "quaternary-700": lambda: _state(700, 300, 4, 7),
    "components": lambda: [[3 * i, 3 * i + 1] for i in range(1500)] + [[3 * i + 1, 3 * i + 2] for i in range(0, 1500, 2)],
    "matching": lambda: [[2 * i, 2 * i + 1] for i in range(800)],
}


@pytest.mark.parametrize("name", list(STATES))
def test_hash_of_a_large_state_equals_oracle(ctx, name):
    st = _dense(STATES[name]())
    want = po.wl_hash(st)
    assert int(ctx.wl_hash([st])[0]) == want
    shuffled = st[:]
    random.Random(11).shuffle(shuffled)
    got = ctx.wl_hash([shuffled, st, st[:300], shuffled])
    assert [int(got[0]), int(got[1]), int(got[3])] == [want] * 3
    assert int(got[2]) == po.wl_hash(_dense(st[:300]))


def test_many_large_states_at_once(ctx):
    sts = [_dense(_state(300 + 7 * (i % 40), 150 + 5 * (i % 31), 2, i)) for i in range(1500)]
    got = ctx.wl_hash(sts)
    for i in range(0, 1500, 13):
        assert int(got[i]) == po.wl_hash(sts[i]), i


LEAF = rule_from_lists([[0, 0]], [[0, 1], [1, 2]])
SWAP3 = rule_from_lists([[0, 1, 0]], [[1, 0, 2]])
EXPAND = {
    "hubs": lambda: Request([LEAF], _hubs(900, [8, 9, 16, 17, 64, 65, 200]) + [[i, i] for i in range(20)], 1, flags=REL),
    "1500-edges": lambda: Request([LEAF], _state(1500, 700, 2, 8) + [[i, i] for i in range(6)], 2, flags=REL),
    "many": lambda: Request([LEAF], _state(250, 300, 2, 10) + [[i, i] for i in range(40)], 2, flags=REL),
    "6000-edges": lambda: Request([LEAF], _state(6000, 9000, 2, 9) + [[i, i] for i in range(6)], 1, flags=REL),
    "9000-edges": lambda: Request([LEAF], _state(9000, 9500, 2, 9) + [[i, i] for i in range(6)], 1, flags=REL),
    "ternary": lambda: Request([SWAP3], _state(1200, 60, 3, 12), 1, flags=REL),
}


@pytest.mark.parametrize("name", list(EXPAND))
def test_large_children_equal_oracle(ctx, name):
    req = EXPAND[name]()
    o = po.evolve(req)
    assert o.counts["events"] > 0
    assert_exact(ctx.evolve(req), o, tr=True)
    if name in ("hubs", "1500-edges", "ternary"):
        try:
            ctx.set_expand_team(2)
            assert np.array_equal(ctx.evolve(req).states()[0], o.state_hash)
        finally:
            ctx.set_expand_team(0)
