"""GPU: a result's arrays as they are read back (states, events, causal pairs with their reduction
tags, causal triples, branchial pairs) equal the oracle's element by element, at the sizes where the
gather can go wrong: no events at all, one event, one past a 256-event workgroup, several roots,
rules of one and of four LHS edges, and arrays longer than one piece of the pinned buffer (131,072
events, 262,144 hashes); and from several threads at once."""
import threading

import numpy as np
import pytest

from hypergraphrewritingengine_amd import workloads as W
from hypergraphrewritingengine_amd.rules import Request, rule_from_lists
from oracle import pyoracle as po
from tests.parity import assert_exact

pytestmark = pytest.mark.gpu

REL = 0x1 | 0x2 | 0x4 | 0x100
SPLIT = rule_from_lists([[0, 1]], [[0, 2], [2, 1]])
QUAD = rule_from_lists([[0, 1], [1, 2], [2, 3], [3, 0]], [[0, 1], [1, 2], [2, 3], [3, 4], [4, 0]])

CASES = {
    "no-steps": lambda: Request([SPLIT], [[0, 1], [1, 2]], 0, flags=REL),
    "no-match": lambda: Request([QUAD], [[0, 1], [1, 2]], 2, flags=REL),
    "one-event": lambda: Request([SPLIT], [[0, 1]], 1, flags=REL),
    "257-events": lambda: Request([SPLIT], [[i, i + 1] for i in range(257)], 1, flags=REL),
    "two-roots": lambda: Request([SPLIT], [[[0, 1], [1, 2]], [[0, 0]]], 4, flags=REL, multi_root=True),
    "four-lhs": lambda: Request([QUAD, SPLIT], [[0, 1], [1, 2], [2, 3], [3, 0]], 3, flags=REL),
    "pieces": lambda: W.config2(5, flags=REL),
}


@pytest.mark.parametrize("name", list(CASES))
def test_arrays_equal_oracle(ctx, name):
    req = CASES[name]()
    assert_exact(ctx.evolve(req), po.evolve(req), tr=True)


def test_results_read_from_several_threads(ctx):
    reqs = [W.config2(4, flags=REL), W.config1(4, flags=REL), CASES["257-events"](), W.config2(5, flags=REL)]
    res = ctx.evolve_batch(reqs)
    want = [(r.states(), r.events(), r.causal(), r.branchial()) for r in res]
    bad = []

    def read(i):
        for _ in range(3):
            got = (res[i].states(), res[i].events(), res[i].causal(), res[i].branchial())
            flat = lambda t: [x for y in t for x in (y if isinstance(y, tuple) else (y,))]  # noqa: E731
            if not all(np.array_equal(a, b) for a, b in zip(flat(got), flat(want[i]))):
                bad.append(i)

    threads = [threading.Thread(target=read, args=(i % 4,)) for i in range(8)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not bad
