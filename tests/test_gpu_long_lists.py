"""GPU: dense states, most of whose neighbour lists are long, against the oracle. Small children: more long
entries than are numbered at once (several batches), lists on both sides of half of them, teams of one wave
with different numbers of batches. Large states: lists around 64 entries and multiples, one list and hundreds."""
import random

import pytest

from hypergraphrewritingengine_amd.rules import Request, rule_from_lists
from oracle import pyoracle as po
from tests.parity import assert_exact
from tests.test_gpu_general_kernels import _ms

pytestmark = pytest.mark.gpu

REL = 0x1 | 0x2 | 0x4 | 0x100
TURN = {2: rule_from_lists([[0, 1]], [[1, 0]]), 3: rule_from_lists([[0, 1, 2]], [[1, 2, 0]]),
        4: rule_from_lists([[0, 1, 2, 3]], [[3, 1, 0, 4]])}


def _dense(m, n, a, seed=0):
    """m edges of arity a over exactly n vertices."""
    rnd = random.Random(1000 * m + n + seed)
    edges = [[rnd.randrange(n) for _ in range(a)] for _ in range(m)]
    for v in range(n):
        edges[v % m][v // m % a] = v
    return edges


def _hubs(degrees, m, n):
    """Hubs of the given degrees on leaves of their own beside a dense part."""
    edges, nxt = _dense(m, n, 2), n
    for d in degrees:
        edges += [[nxt, nxt + 1 + i] if i % 2 else [nxt + 1 + i, nxt] for i in range(d)]
        nxt += d + 1
    return edges


SMALL = [(2, _dense(m, n, 2)) for m, n in ((60, 6), (64, 9), (100, 10), (128, 16), (128, 28), (200, 20), (254, 30), (255, 2),
                                           (255, 4), (255, 10), (250, 60))]
SMALL += [(2, _hubs(d, m, n)) for d, m, n in (([100], 60, 6), ([60, 70], 100, 10), ([110], 130, 12), ([16, 17, 9], 200, 24))]
SMALL += [(3, _dense(m, n, 3)) for m, n in ((20, 12), (64, 60), (100, 12), (255, 100), (255, 6))]
SMALL += [(4, _dense(m, n, 4)) for m, n in ((12, 30), (60, 30), (60, 160), (100, 8), (250, 240), (254, 5))]


def _small(i):
    arity, state = SMALL[i]
    return Request([TURN[arity]], state, 1, flags=REL)


@pytest.mark.parametrize("i", range(len(SMALL)))
def test_small_dense_children_equal_oracle(ctx, i):
    req = _small(i)
    o = po.evolve(req)
    try:
        for lanes in (0, 16, 32, 64):
            ctx.set_expand_lanes(lanes)
            assert_exact(ctx.evolve(req), o, tr=True)
    finally:
        ctx.set_expand_lanes(0)


def test_small_dense_children_side_by_side(ctx):
    reqs = [_small(i) for i in range(len(SMALL))]
    reqs += [Request([TURN[2]], _dense(40 + 3 * k, 4 + k % 13, 2, k), 2, flags=REL, state_cap=600) for k in range(60)]
    want = [po.evolve(r) for r in reqs]
    try:
        for lanes in (0, 16, 32, 64):
            ctx.set_expand_lanes(lanes)
            for r, o in zip(ctx.evolve_batch(reqs), want):
                assert_exact(r, o, tr=True)
    finally:
        ctx.set_expand_lanes(0)


def test_small_dense_children_take_no_longer_than_by_the_general_kernel(ctx):
    """0.44 and 0.16 of it; with one list after another the first took 1.7 times as long."""
    for reqs in ([Request([TURN[2]], _dense(240, 30, 2, k), 1, flags=0x1) for k in range(16)],
                 [Request([TURN[4]], _dense(90, 90, 4, k), 1, flags=0x1) for k in range(40)]):
        batch = ctx.prepare(reqs)
        ctx.evolve_batch(batch)
        own = _ms(ctx, "k_expand", batch)
        try:
            ctx.set_expand_team(1)
            general = _ms(ctx, "k_expand", batch)
        finally:
            ctx.set_expand_team(0)
        print(own, general)
        assert own < general
LARGE = [_dense(m, n, 2) for m, n in ((300, 2), (300, 9), (1200, 9), (2000, 25), (2000, 62), (4000, 64), (12000, 100),
                                      (12000, 200))]
LARGE += [_hubs(d, m, n) for d, m, n in (([63, 64, 65, 66, 127, 128, 129, 130], 300, 100), ([1000, 65], 900, 9),
                                         ([70] * 70, 400, 300), ([64, 4000], 300, 40))]
LARGE += [_dense(900, 20, 3), _dense(900, 40, 3), _dense(700, 10, 4), _dense(700, 60, 4)]


def _compact(edges):
    ids = {}
    return [[ids.setdefault(v, len(ids)) for v in e] for e in edges]


@pytest.mark.parametrize("i", range(len(LARGE)))
def test_large_dense_states_equal_oracle(ctx, i):
    state = _compact(LARGE[i])
    other = state[:]
    random.Random(i).shuffle(other)
    got = ctx.wl_hash([state, other])
    assert [int(x) for x in got] == [po.wl_hash(state)] * 2
    a = len(state[0])
    top = max(v for e in state for v in e)
    req = Request([rule_from_lists([[0] * a], [[0] * a, list(range(a))])],
                  state + [[top + 1 + k] * a for k in range(3)], 1, flags=REL)
    assert_exact(ctx.evolve(req), po.evolve(req), tr=True)


def test_large_dense_children_take_no_longer_than_by_the_general_kernel(ctx):
    """0.6 and 0.2 of it; with one list above 64 entries after another the first took 9 times as long."""
    for m, n in ((2000, 40), (12000, 200)):
        state = _dense(m, n, 2)
        req = Request([rule_from_lists([[0, 0]], [[0, 0], [0, 1]])], state + [[n + k] * 2 for k in range(3)], 1, flags=0x1)
        batch = ctx.prepare([req])
        ctx.evolve_batch(batch)
        own = _ms(ctx, "k_expand", batch)
        try:
            ctx.set_expand_team(8)
            general = _ms(ctx, "k_expand", batch)
        finally:
            ctx.set_expand_team(0)
        print(own, general)
        assert own < general
