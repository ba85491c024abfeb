"""Results read back from plans: downloads of a batch bring the following
sets along and keep pinned memory between calls, so sets are read here in
order, out of order, twice, across runs and from several threads, each
against its own plan's result."""
from concurrent.futures import ThreadPoolExecutor

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def same(a, b):
    assert np.array_equal(a.raw_tally, b.raw_tally)
    assert np.array_equal(a.value, b.value) and np.array_equal(a.count, b.count)
    assert np.array_equal(a.type_count, b.type_count)
    assert a.stats["divisions"] == b.stats["divisions"] and a.stats["lost"] == b.stats["lost"]


@pytest.mark.parametrize("n_sets,order", [(2, "up"), (37, "up"), (37, "down"), (37, "mixed")])
def test_batch_results_in_any_order(procell_lib, n_sets, order):
    from procell import workloads

    ws = workloads.parameter_sets(3, n_sets, scale=0.05)
    probs = [procell_lib.Problem.from_workload(w, 0) for w in ws]
    seeds = np.arange(n_sets, dtype=np.uint64) + 70
    idx = {"up": list(range(n_sets)), "down": list(range(n_sets))[::-1],
           "mixed": [(7 * i) % n_sets for i in range(n_sets)] + [5, 5, 6, 7, 0]}[order]
    with procell_lib.Batch(probs) as batch:
        for shift in (0, 1000):
            s = seeds + np.uint64(shift)
            batch.run(s)
            for i in idx:
                same(batch.result(i), procell_lib.simulate(procell_lib.Problem.from_workload(ws[i], int(s[i]))))


def test_results_from_several_threads(procell_lib):
    from procell import workloads

    ws = workloads.parameter_sets(4, 24, scale=0.05)
    seeds = np.arange(24, dtype=np.uint64)
    refs = [procell_lib.simulate(procell_lib.Problem.from_workload(w, int(s))) for w, s in zip(ws, seeds)]
    with procell_lib.Batch([procell_lib.Problem.from_workload(w, 0) for w in ws]) as batch, \
            ThreadPoolExecutor(4) as pool:
        batch.run(seeds)
        for got, ref in zip(pool.map(batch.result, range(24)), refs):
            same(got, ref)
        # whole calls in parallel, each on a stream of its own
        again = pool.map(lambda k: procell_lib.simulate(procell_lib.Problem.from_workload(ws[k], int(seeds[k]))), range(24))
        for got, ref in zip(again, refs):
            same(got, ref)
