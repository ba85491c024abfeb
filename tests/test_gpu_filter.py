"""The filtered simulation kernel (single-precision times, 64-bit evaluation
of the tests within their error bound) against the oracle: whole numbers, so
every comparison is exact.  Cases sit where its rules and bounds lie: the
ranges of times it takes, times close together and many refused candidates,
type tables around its search's groups, cells around the 64 of a root step,
trees at the limits of 32-bit node indices, rows beyond the tally window."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

STATS = ("divisions", "recorded", "dropped", "lost", "rejected", "cells")


def check(procell, oracle, values, counts, proportion, mean, sd, t_max, phi, seed, **kw):
    res = procell.simulate(procell.Problem(values, counts, proportion, mean, sd, t_max, phi, seed, **kw))
    tally, _, st = oracle.simulate(oracle.Problem(values, counts, proportion, mean, sd, t_max, phi, seed))
    diff = np.argwhere(res.raw_tally != tally)
    assert diff.size == 0, f"{len(diff)} tally entries differ, first {diff[:5].tolist()}"
    assert {k: res.stats[k] for k in STATS} == {k: st[k] for k in STATS}
    return st


# t_max 1e-9 and 1e12 are the last values the filter takes; beyond them, and
# at 0 and infinity, the plan runs the 64-bit kernel
@pytest.mark.parametrize("t_max", [0.9e-9, 1e-9, 1.0, 1e12, 1.1e12])
@pytest.mark.parametrize("spread", [0.0, 1e-3, 0.4, 3.0])
def test_time_scales_and_spreads(procell_lib, oracle, t_max, spread):
    mean = t_max / 4.7
    st = check(procell_lib, oracle, [4000.0, 90.0, 700.0], [9000, 4000, 7001], [0.7, 0.3], [mean, 2.1 * mean],
               [spread * mean, 2.0 * spread * mean], t_max, 3.0, 12)
    assert st["divisions"] > 1000


@pytest.mark.parametrize("n_types", [1, 2, 4, 5, 6, 9, 10, 17, 256])
def test_type_search_groups(procell_lib, oracle, n_types):
    # the last types have proportion 0: the running sum reaches 1 before them
    p = np.zeros(n_types)
    n = max(1, n_types - 2)
    p[:n] = 1.0 / n
    mean = 20.0 + 3.0 * np.arange(n_types) % 50
    check(procell_lib, oracle, [900.0, 33.0], [20000, 3000], p, mean, 0.3 * mean, 80.0, 2.0, 5)


@pytest.mark.parametrize("cells", [1, 63, 64, 65, 127, 513, 4097])
@pytest.mark.parametrize("block", [0, 64, 192])
def test_cells_around_a_root_step(procell_lib, oracle, cells, block):
    check(procell_lib, oracle, [3000.0, 500.0], [cells, 1], [0.6, 0.4], [20.0, -1.0], [6.0, -1.0], 110.0, 1.0, cells,
          block_size=block)


@pytest.mark.parametrize("cap", [0, 1, 2, 30, 31, 32, 45])
def test_generation_caps(procell_lib, oracle, cap):
    # values 1.5 * 2**cap over phi = 1: caps cap and cap + 1 either side of the
    # 32-bit node indices; t_max allows about seven generations
    check(procell_lib, oracle, [1.5 * 2.0 ** cap, 1.5 * 2.0 ** (cap + 1)], [400, 300], [1.0], [10.0], [4.0], 75.0, 1.0, 3)


@pytest.mark.parametrize("rows,per_row", [(40, 700), (3000, 3)])
def test_rows_beyond_the_window(procell_lib, oracle, rows, per_row):
    # one segment over all rows: most tallies go to the device directly
    values = np.geomspace(2.0, 3e4, rows)
    check(procell_lib, oracle, values, [per_row] * rows, [0.5, 0.5], [15.0, 40.0], [5.0, 9.0], 95.0, 1.0, 9,
          segments=1, blocks_per_cu=1, block_size=64)
