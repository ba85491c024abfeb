"""GPU: procell_simulate_noalloc with as many rows as its static scratch holds
without the filtered kernel's row table: the same outputs as procell_simulate,
bit for bit."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows", [300_000, 900_000, 1_040_000])
def test_noalloc_takes_rows_up_to_its_scratch(procell_lib, rows):
    prob = procell_lib.Problem(np.linspace(1.0, 1.9, rows), np.ones(rows), [1.0], [20.0], [5.0], 30.0, 1.0, 3)
    ref, got = procell_lib.simulate(prob), procell_lib.simulate_noalloc(prob)
    assert ref.stats["recorded"] > 0 and ref.stats["dropped"] > 0
    assert np.array_equal(ref.raw_tally, got.raw_tally)
    assert np.array_equal(ref.value, got.value) and np.array_equal(ref.count, got.count)
    for k in ("divisions", "recorded", "dropped", "lost", "rejected", "cells", "pool"):
        assert ref.stats[k] == got.stats[k], k
