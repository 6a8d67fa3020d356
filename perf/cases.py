"""The calls that the framework's speed is measured on.

A case is a dict of plain values; its "kind" names one way in which a program uses the package:

  evolve    one request with host inputs, evolved alone, its arrays read back
  batch     many requests prepared once (device-resident inputs), evolved together, counts read
  relations a batch with host inputs whose states, events and relations are all read back
  replay    a prepared batch's pass as one HIP graph, launched again and again
  serve     requests submitted to the served path, driven until every one has finished
  quotient  quotient exploration of one request and the raw unfolding beneath it
  match     all matches of one rule in one large state held in device memory

Every input is drawn from the seed alone. Where a case's amount of work must not depend on the
seed, a fixed active core (the rule's own start) stands beside a random part that the rule never
matches, so the states differ from seed to seed and the number of events does not.
"""
from __future__ import annotations

import random

import numpy as np
import torch

import hypergraphrewritingengine_amd as hgx
from hypergraphrewritingengine_amd import abi
from hypergraphrewritingengine_amd import workloads as W
from hypergraphrewritingengine_amd.rules import Request, rule_from_lists

REC_CAUSAL, REC_BRANCHIAL, REC_RELATIONS, REC_STATES, OPT_TR = 0x1, 0x2, 0x4, 0x8, 0x100

# rule, active core, and the events of one evolution of the core by step (explored events for wpp)
RULES = {
    # every directed path of two edges gains its closing edge
    "triangle": (([[0, 1], [1, 2]], [[0, 1], [1, 2], [2, 0]]), [[0, 1], [1, 2], [2, 0]], (3, 18, 135, 1464, 22203)),
    # two edges out of one vertex become four: the standard growing rule
    "growth": (([[0, 1], [0, 2]], [[0, 2], [0, 3], [1, 3], [2, 3]]), [[0, 0], [0, 0]],
               (2, 26, 434, 9938, 290018, 10309586)),
    # the Wolfram-physics rule of the published quotient timings
    "wpp": (([[0, 1], [0, 2]], [[0, 1], [0, 3], [1, 3], [2, 3]]), [[0, 1], [0, 2]],
            (2, 4, 12, 52, 400, 3866)),
}

_CTX = None


def _ctx():
    """The one context a program keeps for all of its requests."""
    global _CTX
    if _CTX is None:
        _CTX = hgx.Context(0)
    return _CTX


def _beside(rule, seed, extra, first):
    """`extra` binary edges on vertices from `first` up, disjoint from the core, that no match of the
    rule takes: for the triangle rule from sources to targets (no path of two edges), for the rules
    of two edges out of one vertex a random map (one edge out of each vertex)."""
    rnd = random.Random(seed * 2654435761 + 97)
    if rule == "triangle":
        k = extra // 2 + 1
        return [[first + rnd.randrange(k), first + k + rnd.randrange(k)] for _ in range(extra)]
    return [[first + i, first + rnd.randrange(extra)] for i in range(extra)]


def _core_request(case, seed, flags):
    (lhs, rhs), core, _ = RULES[case["rule"]]
    return Request([rule_from_lists(lhs, rhs)], core + _beside(case["rule"], seed, case["extra"], 8),
                   case["steps"], flags=flags)


def _scan(n, extra):
    """The n evolutions of a relations case: both rules, 3 and 4 steps, 9 to 9 + extra edges beside the core."""
    return [{"rule": ("triangle", "growth")[i % 2], "steps": 3 + i // 2 % 2, "extra": 9 + i * 7 % (extra + 1)}
            for i in range(n)]


def _ints(a):
    """An array of whole numbers in the signed type of its width."""
    return a.view({8: np.int64, 4: np.int32, 2: np.int16, 1: np.int8}[a.dtype.itemsize])


def _counts(rows):
    return {k: _ints(np.ascontiguousarray(rows[k])) for k in rows.dtype.names}


def _everything(r):
    h, step, creator = r.states()
    causal, tr = r.causal()
    return {"hash": _ints(h), "step": _ints(step), "creator": _ints(creator), "events": _ints(r.events()),
            "causal": _ints(causal), "in_tr": _ints(tr), "branchial": _ints(r.branchial())}


def _first(seed):
    """Where a seed's draws of the seeded workloads start."""
    return (seed * 1000003 + 12345) % (1 << 40)


def listed():
    return [
        # the smallest call: an interactive evaluation of a few steps, all of it read back
        {"name": "evolve-small", "kind": "evolve", "rule": "triangle", "steps": 3, "extra": 9, "read": True},
        # a notebook-sized multiway graph with every relation read back for plotting
        {"name": "evolve-readback", "kind": "evolve", "rule": "growth", "steps": 5, "extra": 9, "read": True},
        # one large evolution whose size and canonical count are wanted (ten million raw states)
        {"name": "evolve-large", "kind": "evolve", "rule": "growth", "steps": 6, "extra": 7, "read": False},
        # states of tens of thousands of vertices: one rewriting step of a space-like hypergraph
        {"name": "evolve-wide-states", "kind": "evolve", "rule": "random", "steps": 1, "edges": 12001, "read": True},
        # the benchmark's batch: a rule-space scan from device-resident inputs
        {"name": "batch-4096", "kind": "batch", "n": 4096, "cap": 4096},
        # a small scan, where the launches of a generation hold little work
        {"name": "batch-61", "kind": "batch", "n": 61, "cap": 4096},
        # a scan with host inputs whose relations are all fetched
        {"name": "relations-60", "kind": "relations", "n": 60, "extra": 50},
        # the same batch evaluated repeatedly as one graph launch
        {"name": "replay-1000", "kind": "replay", "n": 1000, "cap": 4096},
        # a burst of service requests with initial states of 3 to 2,048 edges
        {"name": "serve-100", "kind": "serve", "n": 100, "cap": 4096},
        # exploration up to isomorphism with the raw multiway counts beneath it
        {"name": "quotient-6", "kind": "quotient", "rule": "wpp", "steps": 6, "extra": 8},
        # one rewriting step's matches of a large ternary hypergraph, and of a large graph's triangles
        {"name": "match-ternary", "kind": "match", "rule": "ternary", "edges": 50000, "vertices": 10000},
        {"name": "match-triangle", "kind": "match", "rule": "cycle", "edges": 200000, "vertices": 20000},
    ]


def draw(rng):
    def log_int(lo, hi):
        return int(round(lo * (hi / lo) ** rng.random()))

    kind = rng.choice(["evolve", "evolve", "wide", "batch", "batch", "relations", "replay", "serve", "quotient",
                       "match", "match"])
    if kind == "evolve":
        rule = rng.choice(["triangle", "growth"])
        return {"kind": "evolve", "rule": rule, "steps": rng.randint(3, 5), "extra": rng.randint(9, 120),
                "read": rng.random() < 0.5}
    if kind == "wide":
        return {"kind": "evolve", "rule": "random", "steps": 1, "edges": log_int(2500, 12001), "read": True}
    if kind == "batch":
        return {"kind": "batch", "n": log_int(17, 4096), "cap": log_int(256, 4096)}
    if kind == "relations":
        return {"kind": "relations", "n": log_int(7, 60), "extra": rng.randint(0, 50)}
    if kind == "replay":
        return {"kind": "replay", "n": log_int(33, 2000), "cap": log_int(256, 4096)}
    if kind == "serve":
        return {"kind": "serve", "n": log_int(5, 100), "cap": log_int(256, 4096)}
    if kind == "quotient":
        return {"kind": "quotient", "rule": "wpp", "steps": rng.randint(4, 6), "extra": rng.randint(8, 20)}
    rule = rng.choice(["ternary", "cycle"])
    edges = log_int(5000, 50000 if rule == "ternary" else 200000)
    return {"kind": "match", "rule": rule, "edges": edges, "vertices": max(3, edges // (5 if rule == "ternary" else 10))}


# rules of the large-state joins: a ternary wedge, and a directed triangle
MATCH_RULES = {
    "ternary": ([[0, 1, 2], [2, 3, 4]], [[0, 3, 5], [1, 4, 5], [2, 5, 5]]),
    "cycle": ([[0, 1], [1, 2], [2, 0]], [[0, 1], [1, 2], [2, 0], [0, 3]]),
}


def _mean_matches(case):
    """Expected matches of a random state of m edges on n vertices."""
    m, n = case["edges"], case["vertices"]
    return m * m / n if case["rule"] == "ternary" else m ** 3 / n ** 3


def prepare(case, seed):
    kind = case["kind"]
    s = {"case": case, "ctx": _ctx()}
    if kind == "evolve" and case["rule"] == "random":
        # a sparse random acyclic graph, with 120 directed triangles that some of its edges lead to
        rng = np.random.default_rng([seed, 1])
        m = case["edges"]
        source = rng.integers(0, m, size=m - 360)
        edges = np.stack([source, rng.integers(source + 1, m + 360)], axis=1)
        corner = m + np.arange(360).reshape(120, 3)
        edges = np.concatenate([edges, corner[:, [0, 1]], corner[:, [1, 2]], corner[:, [2, 0]]])
        edges = edges[rng.permutation(len(edges))]
        # reverse a directed triangle
        rule = rule_from_lists([[0, 1], [1, 2], [2, 0]], [[0, 2], [2, 1], [1, 0]])
        s["request"] = Request([rule], edges.tolist(), case["steps"],
                               flags=REC_CAUSAL | REC_BRANCHIAL | REC_RELATIONS | OPT_TR)
    elif kind == "evolve":
        flags = REC_CAUSAL | REC_BRANCHIAL | (REC_RELATIONS | OPT_TR if case["read"] else 0)
        s["request"] = _core_request(case, seed, flags)
    elif kind == "quotient":
        s["request"] = _core_request(case, seed, REC_CAUSAL | REC_BRANCHIAL | REC_STATES | OPT_TR |
                                     abi.HGX_OPT_QUOTIENT)
    elif kind in ("batch", "replay"):
        reqs = [W.batched_run(_first(seed) + i, cap=case["cap"]) for i in range(case["n"])]
        s["batch"] = s["ctx"].prepare(reqs)
        if kind == "replay":
            s["replay"] = s["ctx"].capture(s["batch"])
    elif kind == "relations":
        flags = REC_CAUSAL | REC_BRANCHIAL | REC_RELATIONS | OPT_TR
        s["requests"] = [_core_request(c, seed * 4096 + i, flags) for i, c in enumerate(_scan(case["n"], case["extra"]))]
    elif kind == "serve":
        s["requests"] = [W.served_run(_first(seed) + i, cap=case["cap"]) for i in range(case["n"])]
    elif kind == "match":
        rng = np.random.default_rng([seed, 2])
        lhs, rhs = MATCH_RULES[case["rule"]]
        a = len(lhs[0])
        s["rules"] = [rule_from_lists(lhs, rhs)]
        s["vertices"] = torch.from_numpy(rng.integers(0, case["vertices"], size=(case["edges"], a),
                                                      dtype=np.int32)).cuda()
        s["arity"] = torch.full((case["edges"],), a, dtype=torch.uint8, device="cuda")
        s["cap"] = int(1.5 * _mean_matches(case)) + 4096
        s["matches"] = torch.zeros((s["cap"], len(lhs)), dtype=torch.int32, device="cuda")
        torch.cuda.synchronize()
    return s


def run(s):
    case, ctx = s["case"], s["ctx"]
    kind = case["kind"]
    if kind == "evolve":
        res = ctx.evolve_batch([s["request"]])
        out = _counts(res.counts())
        if case["read"]:
            out.update(_everything(res[0]))
        return out
    if kind == "batch":
        return _counts(ctx.evolve_batch(s["batch"]).counts())
    if kind == "replay":
        return _counts(s["replay"].launch().counts())
    if kind == "relations":
        res = ctx.evolve_batch(s["requests"])
        out = _counts(res.counts())
        parts = [_everything(r) for r in res]
        out.update({k: np.concatenate([p[k] for p in parts]) for k in parts[0]})
        return out
    if kind == "serve":
        ids = [ctx.submit(r) for r in s["requests"]]
        done = {}
        while ctx.serve_step():
            done.update(ctx.drain())
        done.update(ctx.drain())
        rows = [done[i].counts for i in ids]
        return {k: np.array([r[k] for r in rows], np.uint64).view(np.int64) for k in rows[0]}
    if kind == "quotient":
        r = ctx.evolve(s["request"])
        h, step, creator = r.states()
        out = {"counts": r.counts["raw_states"], "hash": _ints(h), "step": _ints(step), "creator": _ints(creator),
               "events": _ints(r.events())}
        out.update({"unfold_" + k: v for k, v in r.unfold().items()})
        return out
    n = ctx.match_noalloc(s["rules"], 0, s["vertices"].data_ptr(), s["arity"].data_ptr(), case["edges"],
                          s["vertices"].shape[1], case["vertices"], s["matches"].data_ptr(), s["cap"])
    return {"count": n, "matches": s["matches"]}


# Means of the seeded workloads' draws, per request (4,096 requests from seed 0 up): raw states,
# edges of a state, initial edges. A draw's evolution grows with its cap less than in proportion.
BATCH_STATES, BATCH_EDGES, BATCH_INIT = 554.0, 37.0, 33.0
SERVE_STATES, SERVE_EDGES, SERVE_INIT = 600.0, 90.0, 310.0


def work(case):
    """Least traffic: the initial states read; every raw state's edges formed (10 bytes a binary
    edge, as the next generation's input) and its record (hash, step, creator) and event written;
    relations written where they are asked for. Operations: a colour refinement costs an update
    per edge end and round (about four operations, six rounds)."""
    kind = case["kind"]
    if kind == "match":
        m, a = case["edges"], len(MATCH_RULES[case["rule"]][0][0])
        k = len(MATCH_RULES[case["rule"]][0])
        found = _mean_matches(case)
        # the state read once, an index of (vertex, position) written and read, the matches written
        return {"bytes": m * (4 * a + 1) + 2 * m * a * 4 + found * 4 * k, "flops": m * a * 4 + found * k * a * 2}
    if kind == "evolve" and case["rule"] == "random":
        states, edges, init, rel = 361.0, float(case["edges"]), float(case["edges"]), 16.0
    elif kind in ("evolve", "quotient"):
        _, core, events = RULES[case["rule"]]
        gain = {"triangle": 1, "growth": 2, "wpp": 2}[case["rule"]]
        states = 1.0 + events[case["steps"] - 1]
        init = float(len(core) + case["extra"])
        edges = init + gain * case["steps"]
        rel = 16.0 + 8.0 * (2 + 6) if case.get("read") else 0.0
    elif kind == "relations":
        scan = _scan(case["n"], case["extra"])
        states = sum(1.0 + RULES[c["rule"]][2][c["steps"] - 1] for c in scan)
        init = sum(3.0 + c["extra"] for c in scan)
        edges = init / case["n"] + 5
        rel = 16.0 + 8.0 * 6
    else:
        per, edges, init = (SERVE_STATES, SERVE_EDGES, SERVE_INIT) if kind == "serve" else (BATCH_STATES, BATCH_EDGES,
                                                                                            BATCH_INIT)
        states = case["n"] * per * (case["cap"] / 4096.0) ** 0.7
        rel = 0.0
        init *= case["n"]
    return {"bytes": init * 10 + states * (edges * 10 + 16 + 16 + rel), "flops": states * edges * 2 * 4 * 6}


def exact(case, seed):
    """Every output is a whole number: there is nothing to hold against 64-bit arithmetic."""
    return None
