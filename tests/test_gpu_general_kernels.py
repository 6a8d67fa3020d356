"""GPU: one-arity children and binary states by the general kernels, which a forced team of one wave chooses, at
every lane count: equal to the oracle, and so to the kernels of their own they take otherwise."""
import random

import pytest

from hypergraphrewritingengine_amd import workloads as W
from hypergraphrewritingengine_amd.rules import Request, rule_from_lists
from oracle import pyoracle as po
from tests.parity import assert_exact

pytestmark = pytest.mark.gpu

REL = 0x1 | 0x2 | 0x4 | 0x100


def _state(m, n, a, seed):
    rnd = random.Random(seed)
    return [[rnd.randrange(n) for _ in range(a)] for _ in range(m)]


def _requests():
    path = rule_from_lists([[0, 1], [1, 2]], [[0, 1], [1, 2], [2, 3]])
    ternary = rule_from_lists([[0, 1, 2], [2, 3, 4]], [[0, 3, 5], [1, 4, 5], [2, 5, 5]])
    four = rule_from_lists([[0, 1, 2, 3]], [[3, 1, 0, 4], [4, 4, 1, 0]])
    reqs = [W.batched_run(i, cap=400, flags=REL) for i in range(24)]
    reqs += [Request([path], _state(m, m, 2, m), 2, flags=REL, state_cap=800) for m in (3, 31, 64, 65, 127, 200, 255)]
    reqs += [Request([ternary], _state(m, m, 3, m), 2, flags=REL, state_cap=800) for m in (4, 30, 70)]
    return reqs + [Request([four], _state(m, m, 4, m), 2, flags=REL, state_cap=800) for m in (4, 30, 70)]


def _ms(ctx, name, reqs):
    """Least time of one kernel's launches over a few passes, in ms."""
    best = None
    try:
        for _ in range(4):
            ctx.profile(True)
            ctx.evolve_batch(reqs)
            t = ctx.profile_read()[name]["total_ms"]
            best = t if best is None else min(best, t)
    finally:
        ctx.profile(False)
    return best


@pytest.mark.parametrize("lanes", [0, 16, 32, 64])
def test_one_wave_teams_equal_oracle(ctx, lanes):
    reqs = _requests()
    want = [po.evolve(r) for r in reqs]
    try:
        ctx.set_expand_team(1)
        ctx.set_expand_lanes(lanes)
        ctx.set_join_team(1)
        ctx.set_join_lanes(lanes)
        for r, o in zip(ctx.evolve_batch(reqs), want):
            assert_exact(r, o, tr=True)
    finally:
        ctx.set_expand_team(0)
        ctx.set_expand_lanes(0)
        ctx.set_join_team(0)
        ctx.set_join_lanes(0)


def test_a_forced_team_takes_the_general_kernels(ctx):
    """They take about two and four times as long on a batch of small binary requests."""
    reqs = ctx.prepare([W.batched_run(i, cap=1024) for i in range(1024)])
    ctx.evolve_batch(reqs)
    own = {k: _ms(ctx, k, reqs) for k in ("k_expand", "k_match_count")}
    try:
        ctx.set_expand_team(1)
        ctx.set_expand_lanes(64)
        ctx.set_join_team(1)
        ctx.set_join_lanes(64)
        general = {k: _ms(ctx, k, reqs) for k in own}
    finally:
        ctx.set_expand_team(0)
        ctx.set_expand_lanes(0)
        ctx.set_join_team(0)
        ctx.set_join_lanes(0)
    print(own, general)
    assert all(general[k] > 1.5 * own[k] for k in own)
