"""GPU: the gathered transfers between host and device at the sizes where they can go wrong: initial
states whose arity bytes and vertex words end at, below and above a 4,096-byte transfer and start at odd
addresses (several in one generation), arrays past the largest gathered transfer, and ranges of many
requests in several size classes -- each result the oracle's."""
import pytest

from hypergraphrewritingengine_amd import workloads as W
from hypergraphrewritingengine_amd.rules import Request, rule_from_lists
from oracle import pyoracle as po
from tests.parity import assert_exact

pytestmark = pytest.mark.gpu

REL = 0x1 | 0x2 | 0x4 | 0x100
LOOP = rule_from_lists([[0, 0]], [[0, 1], [1, 0]])
SPLIT = rule_from_lists([[0, 1]], [[0, 2], [2, 1]])


def _chain(m, loops):
    return [[i, i] if i < loops else [i, i + 1] for i in range(m)]


@pytest.mark.parametrize("sizes", [(1, 3, 5), (1023, 1, 1024, 3, 1025), (4095, 2, 4096, 1, 4097), (34000, 7, 9)])
def test_initial_states_of_odd_sizes(ctx, sizes):
    reqs = [Request([LOOP], _chain(m, min(m, 3)), 1, flags=REL) for m in sizes]
    for req, res in zip(reqs, ctx.evolve_batch(reqs)):
        assert_exact(res, po.evolve(req), tr=True)


def test_ranges_of_many_requests_in_several_classes(ctx):
    reqs = [Request([SPLIT], _chain(3 + i % 150, 0), 2, state_cap=200 + i % 60, flags=REL) for i in range(400)]
    reqs[::7] = [W.config1(3, flags=REL)] * len(reqs[::7])
    got = ctx.evolve_batch(reqs)
    for i in list(range(0, 400, 37)) + [398, 399]:
        assert_exact(got[i], po.evolve(reqs[i]), tr=True)
