"""GPU: states whose matches pass 2^32. Every join (bit sets, lists, general) must stop counting and refuse
the generation -- truncated under a cap, out of capacity without one -- and leave the other requests of
the batch as they are alone. The totals lie just above a multiple of 2^32, where a 32-bit sum is small."""
import pytest

from hypergraphrewritingengine_amd import abi
from hypergraphrewritingengine_amd.rules import Request, rule_from_lists
from oracle import pyoracle as po
from tests.parity import assert_exact

pytestmark = pytest.mark.gpu

REL = 0x1 | 0x2 | 0x4 | 0x100
STAR = {k: [[0, i] for i in range(1, k + 1)] for k in (3, 4)}


def _hubs(degrees):
    edges, nxt = [], len(degrees)
    for h, d in enumerate(degrees):
        edges += [[h, nxt + i] for i in range(d)]
        nxt += d
    return edges


def _stars(degrees, k):
    total = 0
    for d in degrees:
        p = 1
        for i in range(k):
            p *= d - i
        total += p
    return total


# state, rules, cap, matches
CASES = {
    # no lane of the widest team holds the cap's worth of matches by itself
    "lists": (_hubs([2049, 14]), [STAR[3]], 20_000_000, _stars([2049, 14], 3)),
    "bits": (_hubs([196, 30]), [STAR[4]] * 3, 100_000_000, 3 * _stars([196, 30], 4)),
    # an edge of another arity: the general join
    "general": (_hubs([2049, 14]) + [[5000, 5001, 5002]], [STAR[3]], 20_000_000, _stars([2049, 14], 3)),
}


def test_totals_lie_above_a_multiple_of_two_to_the_32():
    assert [n % 2 ** 32 for *_, n in CASES.values()] == [136, 105584, 136]


@pytest.mark.parametrize("capped", [True, False])
@pytest.mark.parametrize("name", list(CASES))
def test_generation_is_refused(ctx, name, capped):
    state, lhs, cap, matches = CASES[name]
    assert matches > 2 ** 32
    over = Request([rule_from_lists(p, p) for p in lhs], state, 1, flags=REL, state_cap=cap if capped else 0)
    plain = Request([rule_from_lists(STAR[3], [[0, 1], [1, 2]])], _hubs([5, 4]), 2, flags=REL)
    r, other = ctx.evolve_batch([over, plain])
    print(name, capped, r.counts, r.status(), flush=True)
    assert r.counts["raw_states"] == 1 and r.counts["events"] == 0 and r.counts["steps_done"] == 0
    assert r.counts["truncated"] == (1 if capped else 2)
    assert r.status()[0] == (abi.HGX_OK if capped else abi.HGX_ERR_CAPACITY)
    assert_exact(other, po.evolve(plain), tr=True)


def test_a_cap_just_met_and_just_passed(ctx):
    """Every join under the exact number of matches of a generation, and one below it."""
    for state, lhs in ((_hubs([20, 11]), STAR[3]), (_hubs([90, 80, 150]), STAR[3][:2]),
                       (_hubs([20, 11]) + [[70, 71, 72]], STAR[3])):
        n = _stars([sum(e[0] == h for e in state) for h in range(3) if sum(e[0] == h for e in state) > 2], len(lhs))
        for cap, truncated in ((n + 1, 0), (n, 1)):
            req = Request([rule_from_lists(lhs, lhs)], state, 1, flags=0x1, state_cap=cap)
            r = ctx.evolve(req)
            assert r.counts["truncated"] == truncated and r.counts["events"] == (0 if truncated else n)
