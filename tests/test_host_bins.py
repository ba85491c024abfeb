"""The output bin set (every v / 2^k >= phi, distinct) built by exponent and
mantissa, against the definition, where its rule could go wrong: shared
mantissas, values equal to phi and its powers of two, subnormal phi, rows
below phi and negative values."""
import numpy as np
import pytest


def capacity(values, counts, phi):
    rows = [v for v, c in zip(values, counts) if c]
    phi = phi if phi > 0 else min(rows)
    bins = set()
    for f in rows:
        while f >= phi:
            bins.add(f)
            f = f / 2
    return len(bins)


@pytest.mark.parametrize("values,phi", [
    ([8.0, 16.0, 12.0, 3.0, 6.0], 1.0), ([8.0, 16.0, 12.0, 3.0, 6.0], 1.5), ([8.0, 16.0], 8.0),
    ([5.0, 2.0, -7.0, 0.0, 10.0], 2.5), ([1.0], 0.0), ([1e-307, 3e-308, 7e-307], 2.5e-308),
    ([1e-307, 3e-308, 7e-308], 1e-310), ([4e-324, 8e-324], 4e-324), ([1.75, 1.75, 3.5, 7.0, 1.0], 0.4),
])
def test_capacity_is_the_number_of_distinct_halvings(procell_lib, values, phi):
    counts = [1 + i % 3 for i in range(len(values))]
    prob = procell_lib.Problem(values, counts, [1.0], [10.0], [1.0], 10.0, phi=phi)
    assert prob.output_capacity() == capacity(values, counts, phi)


@pytest.mark.parametrize("seed", range(6))
def test_random_tables(procell_lib, seed):
    rng = np.random.default_rng(seed)
    n = int(rng.integers(1, 400))
    values = np.ldexp(rng.integers(8, 16, n) / 8.0 if seed % 2 else rng.uniform(1.0, 2.0, n), rng.integers(-3, 14, n))
    counts = rng.integers(0, 3, n)
    counts[0] = 1
    phi = float(rng.uniform(0.5, 9.0)) if seed % 3 else float(values[counts > 0].min())
    prob = procell_lib.Problem(values, counts, [1.0], [10.0], [1.0], 10.0, phi=phi)
    assert prob.output_capacity() == capacity(values.tolist(), counts.tolist(), phi)
