"""GPU: quiescent types (mean < 0) whose mean single precision holds only as a
denormal or as -0, against the oracle: quiescent all the same, tallied at
generation 0.  Whole numbers, so every comparison is exact."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mean", [-1.0, -1e-38, -1e-45, -7e-46, -1e-50, -5e-324])
@pytest.mark.parametrize("batch", [False, True])
def test_quiescent_means_of_any_magnitude(procell_lib, oracle, mean, batch):
    args = ([400.0, 90.0, 3.0], [700, 333, 65], [0.45, 0.3, 0.25], [mean, 12.0, 2.0 * mean], [-1.0, 4.0, 0.5], 70.0, 2.0)
    prob = procell_lib.Problem(*args, 9)
    if batch:
        other = procell_lib.Problem([50.0], [100], [1.0], [20.0], [5.0], 60.0, 1.0, 0)
        with procell_lib.Batch([other, prob]) as b:
            b.run([4, 9])
            res = b.result(1)
    else:
        res = procell_lib.simulate(prob)
    tally, _, st = oracle.simulate(oracle.Problem(*args, 9))
    assert tally[:, 0, 0].sum() > 0 and tally[:, 1:, 0].sum() == 0
    assert np.array_equal(res.raw_tally, tally)
    for k in ("divisions", "recorded", "dropped", "lost", "rejected", "cells"):
        assert res.stats[k] == st[k], k
