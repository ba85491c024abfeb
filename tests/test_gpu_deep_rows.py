"""GPU: rows of many generations and types, for which the plan lays out fewer
workgroups per CU and a narrow tally window, against the oracle.  Whole
numbers, so every comparison is exact."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows,per_row,n_types", [(1500, 700, 5), (6000, 400, 5), (50000, 50, 5), (25000, 90, 2), (3000, 300, 12)])
def test_deep_rows_match_oracle(procell_lib, oracle, rows, per_row, n_types):
    mean = np.linspace(35.0, 95.0, n_types)
    if n_types == 5:
        mean[-1] = -1.0
    sd = np.where(mean > 0, 0.25 * mean, -1.0)
    args = (np.geomspace(1.0, 1e4, rows), [per_row] * rows, np.ones(n_types) / n_types, mean, sd, 130.0, 1.0, 6)
    res = procell_lib.simulate(procell_lib.Problem(*args))
    assert res.stats["window_rows"] > 0
    tally, _, st = oracle.simulate(oracle.Problem(*args))
    assert np.array_equal(res.raw_tally, tally)
    for k in ("divisions", "recorded", "dropped", "lost", "rejected", "cells"):
        assert res.stats[k] == st[k], k
