"""GPU: a relaxed plan over so many sets that a pass takes several launches over
the same lane stacks: the sets of the first, the middle and the last segments
equal a small plan of the same sets, in every pass."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def test_passes_of_sixty_thousand_sets(procell_lib):
    import torch

    n, pick = 60_000, [*range(0, 20), *range(49_900, 49_960), *range(59_980, 60_000)]
    rng = np.random.default_rng(4)
    means, seeds = rng.uniform(18.0, 40.0, n), rng.integers(1, 2**40, n)
    values, counts = [9000.0, 40.0], [2, 1]

    def problem(i):
        return procell_lib.Problem(values, counts, [0.7, 0.3], [means[i], -1.0], [0.25 * means[i], -1.0], 100.0, 1.0, int(seeds[i]))

    def passes(idx):
        th = torch.tensor(np.concatenate([[means[i], -1.0, 0.25 * means[i], -1.0, 0.7, 0.3] for i in idx]), device="cuda")
        with procell_lib.RelaxedBatch([problem(i) for i in idx], 0.5) as rp:
            per = rp.h_total // len(idx)
            h, hj = (torch.empty(rp.h_total, dtype=torch.float64, device="cuda") for _ in range(2))
            jac = torch.empty((2, rp.h_total), dtype=torch.float64, device="cuda")
            g = torch.linspace(0.1, 1.0, per, dtype=torch.float64, device="cuda").repeat(len(idx))
            grad = torch.empty_like(th)
            rp.forward(th, h)
            n_exp = rp.expansions()
            rp.backward(th, g, grad)
            assert rp.expansions() == n_exp
            rp.jacobian(th, hj, jac)
            assert rp.expansions() == n_exp
        return [x.cpu().numpy() for x in (h.reshape(len(idx), per), hj.reshape(len(idx), per),
                                          jac.reshape(2, len(idx), per).transpose(0, 1), grad.reshape(len(idx), 6))]

    print("60,000 sets", flush=True)
    many, few = passes(range(n)), passes(pick)
    for a, b in zip(many, few):
        assert np.abs(b).max() > 0.1
        np.testing.assert_allclose(a[pick], b, rtol=1e-11, atol=1e-12 * np.abs(b).max())
