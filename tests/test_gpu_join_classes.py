"""GPU: a generation whose size classes change between the join's two passes. Above 32,768 small states the
classes up to 128 edges are separate launches; when most of those states belong to requests that pass their
cap, few are left to emit. A state must be emitted as it was counted: the kernels of binary states leave no
counts per seed behind, which the general join of a mixed class reads."""
import pytest

from hypergraphrewritingengine_amd.rules import Request, rule_from_lists
from oracle import pyoracle as po
from tests.parity import assert_exact

pytestmark = pytest.mark.gpu

REL = 0x1 | 0x2 | 0x4 | 0x100
GROW = rule_from_lists([[0, 1], [0, 2]], [[0, 2], [0, 3], [1, 3], [2, 3]])
TRIANGLE = rule_from_lists([[0, 1], [1, 2]], [[0, 1], [1, 2], [2, 0]])
MIXED = rule_from_lists([[0, 1, 2]], [[0, 1], [1, 2, 3]])


def _requests(steps):
    # 9,504 states each when the fifth generation is counted; its 280,080 children pass the cap
    capped = [Request([GROW], [[0, 0], [0, 0]], steps, flags=REL, state_cap=20000) for _ in range(4)]
    binary = [Request([TRIANGLE], [[0, 1], [1, 2], [2, 0]], steps, flags=REL),
              Request([TRIANGLE], [[0, 1], [1, 2]], steps, flags=REL)]
    mixed = [Request([MIXED], [[0, 1, 2]] + [[i, i + 1] for i in range(3, 3 + extra)], steps, flags=REL)
             for extra in (40, 70)]
    return capped, binary, mixed


def test_requests_that_stop_between_count_and_emit(ctx):
    capped, binary, mixed = _requests(5)
    want = {id(r): po.evolve(r) for r in (capped[0], *binary, *mixed)}
    over = want[id(capped[0])]
    assert over.counts["truncated"] == 1 and over.counts["steps_done"] == 4
    frontier = [sum(int(s) == 4 for s in want[id(r)].state_step) for r in (capped[0], *binary, *mixed)]
    assert 4 * frontier[0] + sum(frontier[1:]) >= 32768 > sum(frontier[1:])
    reqs = [capped[0], binary[0], mixed[0], capped[1], mixed[1], capped[2], binary[1], capped[3]]
    for r, req in zip(ctx.evolve_batch(reqs), reqs):
        assert_exact(r, want.get(id(req), over), tr=True)
