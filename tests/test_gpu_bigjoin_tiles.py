"""The large-state join where its index, its tiles and its closing edges can go wrong: sizes around
a wave, a workgroup and a tile, lists and tuples long enough for the bit-set order, positions that
hold several arities, closing edges first, last, twice and in many copies, states past the size
whose lists are sorted, and a fixed scratch the frontier outgrows -- against the oracle's match
list, in its order."""
import importlib.util
import os

import numpy as np
import pytest

import hypergraphrewritingengine_amd as hgx
from hypergraphrewritingengine_amd.rules import rule_from_lists
from oracle import pyoracle as po

pytestmark = pytest.mark.gpu

_spec = importlib.util.spec_from_file_location(
    "_no_alloc", os.path.join(os.path.dirname(os.path.abspath(__file__)), "test_zz_no_alloc.py"))
_no_alloc = importlib.util.module_from_spec(_spec)
_spec.loader.exec_module(_no_alloc)

WEDGE, TRIANGLE = [[0, 1], [1, 2]], [[0, 1], [1, 2], [2, 0]]
PAIR, LOOP = [[0, 1], [1, 0]], [[0, 0], [0, 1]]
SQUARE = [[0, 1], [1, 2], [2, 3], [3, 0]]                    # two depths, then a closing edge
DIAMOND = [[0, 1], [1, 2], [2, 0], [0, 2]]                   # a closing edge inside, and one last
TWICE = [[0, 1], [0, 1], [1, 2]]                             # a closing edge first
MIXED = [[0, 1, 1], [1, 2], [1, 2, 3], [3, 0]]               # one position, two arities
APART = [[0, 1], [2, 3], [3, 2]]                             # no shared variable, then closing


def _same(ctx, lhs, edges, cap=10**7):
    rule = rule_from_lists(lhs, [[0]])
    n, m, _ = ctx.match([rule], 0, edges, want_edges=True, cap=cap)
    on, om = po.match([rule], 0, edges, want_edges=True, cap=cap)
    assert n == on and np.array_equal(m, om), lhs
    return n


def _random(rng, m, nv, arities=(2,)):
    return [rng.integers(0, nv, int(rng.choice(arities))).tolist() for _ in range(m)]


@pytest.mark.parametrize("m", [1, 2, 63, 64, 65, 255, 256, 257, 1023, 1025, 2049])
def test_sizes_around_waves_workgroups_and_tiles(ctx, m):
    rng = np.random.default_rng(m)
    for lhs in (WEDGE, TRIANGLE, PAIR, LOOP, SQUARE, DIAMOND, TWICE):
        _same(ctx, lhs, _random(rng, m, max(2, m // 4)))
    _same(ctx, MIXED, _random(rng, m, max(2, m // 6), (1, 2, 3)))
    if m <= 257:
        _same(ctx, APART, _random(rng, m, max(2, m // 4)))


@pytest.mark.parametrize("copies", [31, 32, 33, 34, 35, 64, 255, 256, 257, 700])
def test_long_lists_and_repeated_tuples(ctx, copies):
    """A hub listed `copies` times, and one closing tuple in `copies` copies."""
    rng = np.random.default_rng(copies)
    hub = [[0, 1 + int(x)] for x in rng.integers(0, 50, copies)]
    rest = _random(rng, 300, 60)
    mixed = [(hub + rest)[i] for i in rng.permutation(len(hub) + 300)]
    for lhs in (WEDGE, TRIANGLE, TWICE):
        _same(ctx, lhs, mixed)
    tuples = [[70, 71]] * 3 + [[71, 72]] * 5 + [[72, 70]] * copies + rest
    tuples = [tuples[i] for i in rng.permutation(len(tuples))]
    for lhs in (TRIANGLE, PAIR, DIAMOND):
        n = _same(ctx, lhs, tuples)
        assert lhs != TRIANGLE or n >= 3 * 15 * copies
        _same(ctx, lhs, tuples, cap=max(1, n // 3))


@pytest.mark.parametrize("m", [(1 << 20) - 1, (1 << 20) + 1])
def test_both_sides_of_the_sorted_index(ctx, m):
    rng = np.random.default_rng(5)
    ev = rng.integers(0, m, (m, 2))
    ev[rng.integers(0, m, 600), 0] = 7                       # one long list
    edges = ev.tolist()
    assert _same(ctx, WEDGE, edges) > m // 2
    _same(ctx, TRIANGLE, edges)


def test_a_frontier_past_the_fixed_scratch():
    """Sparse lists (partials without candidates past what a tile stages) and splits of the
    frontier in the fixed scratch give the list of the roomy join."""
    ctx, dev = hgx.Context(0), _no_alloc._Dev()
    rng = np.random.default_rng(3)
    try:
        m = 150_000
        ev = rng.integers(0, 12_000, (m, 2))
        ev[:, 0] = ev[:, 0] // 40 * 40                       # few tails: most lists are empty
        edges = ev.tolist()
        d_ev, d_ar, nv = _no_alloc._on_device(dev, edges, 2)
        for lhs in ([[0, 1], [1, 2], [2, 3]], SQUARE):
            rule = rule_from_lists(lhs, [[0]])
            ref_n, ref, _ = ctx.match([rule], 0, edges, want_edges=True, cap=3 * 10**6)
            cap = min(ref_n, 3 * 10**6)
            out = dev.fill(cap * len(lhs) * 4, 0xFF)
            args = ([rule], 0, d_ev, d_ar, m, 2, nv)
            assert ctx.match_noalloc(*args, out, cap) == ref_n
            assert np.array_equal(dev.get(out, cap * len(lhs), np.uint32).reshape(-1, len(lhs)), ref[:cap])
            assert ctx.match_noalloc(*args) == ref_n
    finally:
        dev.free()
        ctx.close()
