"""GPU: large one-arity states on both sides of where the distinct-count table tightens (the LDS no longer holds
the wider one) and of where the colours no longer fit, against the oracle."""
import random

import pytest

from hypergraphrewritingengine_amd.rules import Request, rule_from_lists
from oracle import pyoracle as po
from tests.parity import assert_exact

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("labels", [9900, 11000, 11631, 11632, 12000, 12600, 12716, 12717, 12800])
def test_states_around_the_limits(ctx, labels):
    rnd = random.Random(labels)
    order = list(range(labels))
    rnd.shuffle(order)
    edges = [[order[i], order[i + 1]] for i in range(labels - 1)]
    # (few colours, each of many vertices, and all of them different)
    ring = edges + [[order[-1], order[0]]]
    hair = edges[: labels // 2] + [[order[rnd.randrange(labels // 2)], order[i]] for i in range(labels // 2, labels)]
    got = ctx.wl_hash([edges, ring, hair])
    assert [int(x) for x in got] == [po.wl_hash(s) for s in (edges, ring, hair)]
    req = Request([rule_from_lists([[0, 0]], [[0, 1]])], hair[: labels - 60] + [[i, i] for i in range(3)], 1, flags=0x107)
    assert_exact(ctx.evolve(req), po.evolve(req), tr=True)
