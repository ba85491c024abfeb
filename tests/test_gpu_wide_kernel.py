"""GPU: the 64-bit simulation kernel against the oracle: heap indices of 32 and
64 bits, row tables in LDS and in device memory, type tables around its
search's groups, rows beyond the tally window, lane stacks in device memory,
infinite t_max.  Times are in units that the filtered kernel's bound does not
cover.  Whole numbers, so every comparison is exact."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

STATS = ("divisions", "recorded", "dropped", "lost", "rejected", "cells")
WIDE = (64, 128, 192, 256)  # threads of a workgroup (the filtered kernel's: 512)


def check(res, oracle, args, seed):
    tally, _, st = oracle.simulate(oracle.Problem(*args, seed))
    diff = np.argwhere(res.raw_tally != tally)
    assert diff.size == 0, f"{len(diff)} tally entries differ, first {diff[:5].tolist()}"
    assert {k: res.stats[k] for k in STATS} == {k: st[k] for k in STATS}
    return st


def wide(procell, oracle, args, seed, **kw):
    res = procell.simulate(procell.Problem(*args, seed, **kw))
    assert res.stats["block_size"] in WIDE
    return check(res, oracle, args, seed)


@pytest.mark.parametrize("n_types", [1, 2, 4, 5, 6, 9, 10, 17, 256])
def test_wide_kernel_type_search(procell_lib, oracle, n_types):
    p = np.zeros(n_types)
    n = max(1, n_types - 2)
    p[:n] = 1.0 / n
    mean = (20.0 + 3.0 * np.arange(n_types) % 50) * 1e11
    wide(procell_lib, oracle, ([900.0, 33.0], [20000, 3000], p, mean, 0.3 * mean, 80.0e11, 2.0), 5)


@pytest.mark.parametrize("cap", [0, 1, 2, 30, 31, 32, 45])
def test_wide_kernel_generation_caps(procell_lib, oracle, cap):
    wide(procell_lib, oracle, ([1.5 * 2.0**cap, 1.5 * 2.0 ** (cap + 1)], [400, 300], [1.0], [10.0e11], [4.0e11], 75.0e11, 1.0), 3)


@pytest.mark.parametrize("rows,per_row", [(40, 700), (3000, 3)])  # row tables in LDS, in device memory
def test_wide_kernel_rows_beyond_the_window(procell_lib, oracle, rows, per_row):
    args = (np.geomspace(2.0, 3e4, rows), [per_row] * rows, [0.5, 0.5], [15.0e11, 40.0e11], [5.0e11, 9.0e11], 95.0e11, 1.0)
    wide(procell_lib, oracle, args, 9, segments=1, blocks_per_cu=1, block_size=64)


@pytest.mark.parametrize("cells", [1, 63, 64, 65, 127, 513, 4097])
def test_wide_kernel_infinite_time(procell_lib, oracle, cells):
    args = ([300.0, 50.0], [cells, 1], [0.6, 0.4], [20.0, -1.0], [6.0, -1.0], float("inf"), 1.0)
    st = wide(procell_lib, oracle, args, cells)
    assert st["dropped"] > 0


def test_wide_kernel_batch(procell_lib, oracle):
    args = [([1500.0 + i, 90.0], [60 + i, 41], [0.6, 0.4], [50e11, 70e11], [20e11, 9e11], 240.0e11, 1.0) for i in range(5)]
    args.append(([2.0**34], [40], [1.0], [20e11], [5e11], 130.0e11, 1.0))
    seeds = list(range(70, 76))
    with procell_lib.Batch([procell_lib.Problem(*a, 0) for a in args]) as b:
        b.run(seeds)
        for i, a in enumerate(args):
            res = b.result(i)
            assert res.stats["block_size"] in WIDE
            check(res, oracle, a, seeds[i])
