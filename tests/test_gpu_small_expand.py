"""GPU: children of one arity up to 255 edges and 255 vertex labels (k_expand_small) against the
oracle, and against the general expansion (two waves per child), at every lane count: neighbour lists
of 8, 9 and more entries, lists longer than the entries numbered in LDS (one vertex holding every
edge), many long lists at once, arities 2 to 4, disconnected states, an emptied state, and both
limits and one past them."""
import numpy as np
import pytest

from hypergraphrewritingengine_amd import workloads as W
from hypergraphrewritingengine_amd.rules import Request, rule_from_lists
from oracle import pyoracle as po
from tests.parity import assert_exact

pytestmark = pytest.mark.gpu

REL = 0x1 | 0x2 | 0x4 | 0x100
LEAF = rule_from_lists([[0, 1]], [[0, 1], [0, 2]])
LEAF3 = rule_from_lists([[0, 1, 2]], [[0, 1, 2], [2, 1, 3]])
LEAF4 = rule_from_lists([[0, 1, 2, 3]], [[0, 1, 2, 3], [3, 1, 0, 4]])
DROP = rule_from_lists([[0, 1]], [])
JOIN3 = rule_from_lists([[0, 1], [1, 2], [2, 3]], [[0, 2], [2, 4], [4, 3]])


def _star(m):
    return [[0, i + 1] for i in range(m)]


def _complete(n):
    return [[i, j] for i in range(n) for j in range(n) if i != j]


CASES = {
    **{f"star-{m}": (lambda m=m: Request([LEAF], _star(m), 1, flags=REL)) for m in (7, 8, 9, 63, 64, 127, 128, 250, 254)},
    **{f"loops-{m}": (lambda m=m: Request([LEAF], [[0, 0]] * m, 1, flags=REL)) for m in (4, 5, 60, 130, 254)},
    "path-254-labels": lambda: Request([LEAF], [[i, i + 1] for i in range(253)], 1, flags=REL),
    "path-255-labels": lambda: Request([LEAF], [[i, i + 1] for i in range(254)], 1, flags=REL),
    "255-edges": lambda: Request([rule_from_lists([[0, 1]], [[1, 0]])], [[i % 16, (i * 7) % 16] for i in range(255)], 1,
                                 flags=REL),
    "256-edges": lambda: Request([rule_from_lists([[0, 1]], [[1, 0]])], [[i % 16, (i * 7) % 16] for i in range(256)], 1,
                                 flags=REL),
    "complete-8": lambda: Request([LEAF], _complete(8), 1, flags=REL),
    "complete-15": lambda: Request([LEAF], _complete(15), 1, flags=REL),
    "ternary": lambda: Request([LEAF3], [[i % 5, (i * 3) % 7, i % 11] for i in range(40)], 2, flags=REL, state_cap=1700),
    "ternary-one-vertex": lambda: Request([LEAF3], [[0, 0, 0]] * 60, 1, flags=REL),
    "quaternary": lambda: Request([LEAF4], [[i % 5, (i * 3) % 7, i % 11, 2] for i in range(30)], 1, flags=REL),
    "components": lambda: Request([LEAF], [[3 * i, 3 * i + 1 + i % 2] for i in range(40)] + [[200, 200]], 1, flags=REL),
    "emptied": lambda: Request([DROP], [[0, 1], [1, 2]], 2, flags=REL),
    "three-lhs": lambda: Request([JOIN3, LEAF], W._connected_init(W.Stream(5), 24), 2, flags=REL, state_cap=3000),
}


@pytest.mark.parametrize("name", list(CASES))
def test_small_children_equal_oracle_at_every_lane_count(ctx, name):
    req = CASES[name]()
    o = po.evolve(req)
    try:
        for lanes in (0, 16, 32, 64):
            ctx.set_expand_lanes(lanes)
            assert_exact(ctx.evolve(req), o, tr=True)
        ctx.set_expand_lanes(0)
        ctx.set_expand_team(2)
        assert np.array_equal(ctx.evolve(req).states()[0], o.state_hash)
    finally:
        ctx.set_expand_lanes(0)
        ctx.set_expand_team(0)


def test_small_children_of_all_kinds_in_one_batch(ctx):
    """Teams of one wave with different states side by side, arities mixed over the launch's stride."""
    reqs = [f() for f in CASES.values()] + [W.batched_run(i, cap=512, flags=REL) for i in range(24)]
    want = [po.evolve(r) for r in reqs]
    try:
        for lanes in (0, 16, 32, 64):
            ctx.set_expand_lanes(lanes)
            for r, o in zip(ctx.evolve_batch(reqs), want):
                assert_exact(r, o, tr=True)
    finally:
        ctx.set_expand_lanes(0)
