"""GPU: the relaxed passes at a proportion that is not a number (an optimiser
that has diverged): every entry that a row's walks of that type record in is
not a number, also where the records are exactly 0 (every cell divides in
time, so the sigmoid is 1 and generation 0 holds 0); other types' entries and
those past the generation cap keep their values."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows,per_row", [(5, 40), (1500, 2)])  # within the LDS window, and beyond it
def test_nan_proportion_reaches_zero_entries(procell_lib, oracle, rows, per_row):
    import torch

    values, counts = np.geomspace(1.5, 900.0, rows), [per_row] * rows
    args = (values, counts, [0.5, 0.3, 0.2], [20.0, 31.0, -1.0], [2.0, 4.0, -1.0], 200.0, 2.0, 5)
    prob = procell_lib.Problem(*args)
    ref, _ = oracle.relaxed(oracle.Problem(*args), 0.5)
    deep = values > 8.0
    assert (ref[deep, 0, 0] == 0).all() and (ref[:, :, 1] > 0).any()
    th = torch.tensor([args[3], args[4], args[2]], dtype=torch.float64, device="cuda")
    th[2, 0] = float("nan")
    with procell_lib.Relaxed(prob, 0.5) as rp:
        h, hj = (torch.empty(rp.shape, dtype=torch.float64, device="cuda") for _ in range(2))
        jac = torch.empty((2,) + tuple(rp.shape), dtype=torch.float64, device="cuda")
        rp.forward(th, h)
        rp.jacobian(th, hj, jac)
        h, hj, jac = h.cpu().numpy(), hj.cpu().numpy(), jac.cpu().numpy()
    phi = values >= 2.0
    for x in (h, hj, jac[0], jac[1]):
        assert np.isnan(x[phi, 0, 0]).all()
        assert np.isnan(x[:, :, 0][ref[:, :, 0] > 0]).all()
        assert np.isfinite(x[:, :, 1:]).all() and np.isfinite(x[~phi, 0, 0]).all()
    for x in (h, hj):
        assert np.abs(x[:, :, 1:] - ref[:, :, 1:]).max() <= 1e-10 * ref.max()
