"""GPU: a generation's per-run totals, summed by chunks of 512 states, decide caps and sizes: runs of
one state, runs that end inside, at and past a chunk, many runs in one group of 64 states, and runs
that match nothing give the oracle's counts, each as alone."""
import pytest

from hypergraphrewritingengine_amd.rules import Request, rule_from_lists
from oracle import pyoracle as po

pytestmark = pytest.mark.gpu

SPLIT = rule_from_lists([[0, 1]], [[0, 2], [2, 1]])


def _path(m, steps, cap=0):
    return Request([SPLIT], [[i, i + 1] for i in range(m)], steps, state_cap=cap, flags=0x3)


@pytest.mark.parametrize("sizes", [[1] * 130, [1, 63, 64, 65, 1, 1], [511, 1, 512, 513], [700, 2, 0, 3, 0, 600]])
def test_totals_of_mixed_runs(ctx, sizes):
    # a path of m edges has m children after one step, and their frontier is m states of one run
    reqs = [_path(m, 2, cap=0 if m < 100 else 2000) if m else
            Request([rule_from_lists([[0, 0]], [[0, 1]])], [[0, 1]], 2, flags=0x3) for m in sizes]
    res = ctx.evolve_batch(reqs)
    want = {}
    for m, r, req in zip(sizes, res, reqs):
        if m not in want:
            want[m] = dict(po.evolve(req).counts)
        assert dict(r.counts) == want[m], m
