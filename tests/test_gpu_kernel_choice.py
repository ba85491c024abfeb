"""GPU: the filtered simulation kernel on sets that it would not take alone
(many refused timers, timers below its error bound, timers all alike), against
the oracle: in a batch whose other sets cost far more.  Whole numbers, so
every comparison is exact."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

STATS = ("divisions", "recorded", "dropped", "lost", "rejected", "cells")
FILTERED = 512  # threads of a workgroup


def check(res, oracle, args, seed):
    tally, _, st = oracle.simulate(oracle.Problem(*args, seed))
    diff = np.argwhere(res.raw_tally != tally)
    assert diff.size == 0, f"{len(diff)} tally entries differ, first {diff[:5].tolist()}"
    assert {k: res.stats[k] for k in STATS} == {k: st[k] for k in STATS}
    return st


def two(mean, sd):
    return [0.6, 0.4], [mean, 1.3 * mean], [sd * mean, sd * 1.3 * mean]


HARD = {
    "spread 0.6": ([1500.0, 90.0], [60, 41], *two(30.0, 0.6), 240.0, 1.0),
    "spread 1": ([1500.0, 90.0], [60, 41], *two(40.0, 1.0), 240.0, 1.0),
    "spread 3": ([1500.0, 90.0], [200, 41], *two(50.0, 3.0), 240.0, 1.0),
    "spread 20": ([1500.0, 90.0], [2000, 400], *two(50.0, 20.0), 240.0, 1.0),
    "timers below the bound": ([1500.0, 90.0], [3, 2], *two(5e-4, 0.25), 240.0, 1.0),
    "timers about the bound": ([1500.0, 90.0], [3, 2], *two(2e-3, 0.4), 240.0, 1.0),
    "all alike": ([1500.0, 90.0], [300, 41], *two(30.0, 0.0), 240.0, 1.0),
    "nearly alike": ([1500.0, 90.0], [300, 41], *two(30.0, 1e-5), 240.0, 1.0),
    "deep": ([2.0**34], [60], *two(20.0, 0.4), 130.0, 1.0),
}


@pytest.mark.parametrize("deep", [False, True])  # lane stacks in LDS, in device memory
def test_filtered_kernel_on_hard_sets(procell_lib, oracle, deep):
    sets = {k: v for k, v in HARD.items() if deep or k != "deep"}
    args = list(sets.values()) + [(np.geomspace(4.0, 1500.0, 300), [3000] * 300, *two(45.0, 0.25), 240.0, 1.0)]
    seeds = [50 + i for i in range(len(args))]
    print("hard sets, deep", deep, flush=True)
    with procell_lib.Batch([procell_lib.Problem(*a, 0) for a in args]) as b:
        b.run(seeds)
        for i, name in enumerate(sets):
            res = b.result(i)
            assert res.stats["block_size"] == FILTERED
            st = check(res, oracle, args[i], seeds[i])
            assert st["divisions"] > 100, name
            if name.startswith("spread"):
                assert st["rejected"] > 50, name
