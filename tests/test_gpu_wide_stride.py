"""GPU: small one-arity requests beside one of arity 5 or more, whose edges set the stride of the whole
generation: the expansion, joins and hashes of the small ones over strides they are not laid out for."""
import random

import pytest

from hypergraphrewritingengine_amd.rules import Request, rule_from_lists
from oracle import pyoracle as po
from tests.parity import assert_exact

pytestmark = pytest.mark.gpu

REL = 0x1 | 0x2 | 0x4 | 0x100


def _small(arity, steps):
    rnd = random.Random(arity)
    lhs = [list(range(arity)), [arity - 1] + list(range(arity, 2 * arity - 1))]
    rhs = [list(range(arity)), [0] + list(range(2 * arity - 1, 3 * arity - 2))]
    return Request([rule_from_lists(lhs, rhs)], [[rnd.randrange(4) for _ in range(arity)] for _ in range(8)], steps,
                   flags=REL, state_cap=3000)


def _wide(arity, edges):
    rnd = random.Random(edges)
    state = [[rnd.randrange(edges) for _ in range(arity)] for _ in range(edges - 1)] + [[7] * arity]
    return Request([rule_from_lists([[0] * arity], [[0] * arity, list(range(arity))])], state, 3, flags=REL)


@pytest.mark.parametrize("wide", [4, 5, 6, 8])
@pytest.mark.parametrize("edges", [140, 600])
def test_one_wide_request_in_the_batch(ctx, wide, edges):
    reqs = [_small(2, 3), _small(3, 3), _wide(wide, edges), _small(4, 2), _small(2, 4)]
    for r, req in zip(ctx.evolve_batch(reqs), reqs):
        assert_exact(r, po.evolve(req), tr=True)


@pytest.mark.parametrize("edges", [140, 600])
def test_large_one_arity_states_beside_a_wide_request(ctx, edges):
    rnd = random.Random(edges)
    state = [[rnd.randrange(edges // 2), rnd.randrange(edges // 2)] for _ in range(edges)]
    large = Request([rule_from_lists([[0, 1], [1, 0]], [[0, 0], [1, 1]])], state, 2, flags=REL)
    reqs = [large, _wide(6, edges), _small(2, 3)]
    for r, req in zip(ctx.evolve_batch(reqs), reqs):
        assert_exact(r, po.evolve(req), tr=True)
