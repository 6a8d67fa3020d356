"""The benchmark's comparison with the CPU baseline: a run that its cap stopped is compared by its counts up to
the generation it completed, and a wrong count is a mismatch."""
import bench
from hypergraphrewritingengine_amd import workloads as W
from oracle import pyoracle as po


def test_capped_runs_agree_and_a_wrong_count_does_not():
    reqs = [W.batched_run(i, cap=200) for i in range(12)]
    counts = [dict(po.evolve(r).counts) for r in reqs]
    assert {c["truncated"] for c in counts} == {0, 1}
    assert bench.cpu_baseline(reqs, counts, 60.0, 1)["count_mismatches"] == 0
    counts[3]["causal_pairs"] += 1
    counts[7]["fingerprint"] ^= 1
    assert bench.cpu_baseline(reqs, counts, 60.0, 1)["count_mismatches"] == 2
