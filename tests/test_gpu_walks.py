"""GPU: the walk kernel of the relaxed estimator at the sizes where it can go
wrong, against the oracle.

Forward pass, adjoint and Jacobian pass (contracted with the adjoint's
cotangent) within the tolerances of the relaxed parity tests: FP64 sums in
another order, and a square root and a reciprocal of at most one unit in the
last place.  Proliferating types per cell around the divisors and multiples
of a wavefront's 64 lanes; one cell; rows of one cell, of which a root step
with a cell stride passes more than 64; rows beyond the window; timers often
<= 0 (redraws beside other lanes' expansions); trees deeper than 31
generations (64-bit heap indices); a single deep walk (shared lanes).
"""
import numpy as np
import pytest

from test_gpu_relaxed import G_ATOL, G_RTOL, H_ATOL, H_RTOL, _args

pytestmark = pytest.mark.gpu


def _case(seed, rows, cells, prolif, quiet, t_max, top=1e4, sd=0.25, mean=(25.0, 60.0)):
    rng = np.random.default_rng(seed)
    m = list(rng.uniform(mean[0], mean[1], prolif)) + [-1.0] * quiet
    s = [sd * x if x > 0 else -1.0 for x in m]
    p = rng.dirichlet(np.ones(len(m)))
    return dict(values=np.geomspace(1.5, top, rows) if rows > 1 else [top], counts=rng.multinomial(cells - rows, np.ones(rows) / rows) + 1,
                proportion=p / p.sum(), mean=m, sd=s, t_max=t_max, phi=1.0, seed=seed)


CASES = {
    "one cell": (_case(1, 1, 1, 1, 0, 150.0), 1),
    "3 types": (_case(2, 7, 1000, 3, 1, 140.0), 1),
    "33 types": (_case(3, 5, 67, 33, 0, 110.0), 1),
    "64 types": (_case(4, 3, 41, 64, 1, 100.0), 2),
    "65 types": (_case(5, 3, 41, 65, 0, 100.0), 1),
    "rows of one cell, stride 16": (_case(6, 4000, 4000, 1, 1, 110.0), 16),
    "rows beyond the window": (_case(7, 2000, 2500, 3, 1, 90.0), 1),
    "redraws": (_case(8, 9, 3000, 2, 0, 60.0, top=300.0, sd=0.7, mean=(20.0, 40.0)), 1),
    "64-bit indices": (_case(9, 4, 300, 2, 0, 150.0, top=2.0**36), 1),
    "one deep walk": (_case(10, 1, 1, 1, 0, 260.0, top=2.0**20, mean=(20.0, 20.1)), 1),
    "quiescent only": (_case(11, 30, 500, 0, 2, 50.0), 4),
}


@pytest.mark.parametrize("name", CASES)
def test_walks_match_oracle(procell_lib, oracle, name):
    import torch

    d, stride = CASES[name]
    beta = 0.5
    print("walks:", name, flush=True)
    op = oracle.Problem(*_args(d))
    h_ref, _ = oracle.relaxed(op, beta)
    g = np.random.default_rng(50).normal(size=h_ref.shape)
    _, grad_ref = oracle.relaxed(op, beta, g)
    th = torch.tensor(np.stack([d["mean"], d["sd"], d["proportion"]]), dtype=torch.float64, device="cuda")
    gt = torch.tensor(g, dtype=torch.float64, device="cuda")
    h, hj, grad, gj = np.zeros_like(h_ref), np.zeros_like(h_ref), np.zeros(th.shape), np.zeros(th.shape)
    with procell_lib.Relaxed(procell_lib.Problem(*_args(d)), beta) as rp:
        o, oj = (torch.empty(rp.shape, dtype=torch.float64, device="cuda") for _ in range(2))
        jac = torch.empty((2,) + tuple(rp.shape), dtype=torch.float64, device="cuda")
        og = torch.empty_like(th)
        for phase in range(stride):
            rp.set_stride(stride, phase)
            rp.forward(th, o)
            n = rp.expansions()
            rp.backward(th, gt, og)
            assert rp.expansions() == n
            rp.jacobian(th, oj, jac)
            assert rp.expansions() == n
            h += o.cpu().numpy()
            hj += oj.cpu().numpy()
            grad += og.cpu().numpy()
            gj[:2] += (gt * jac).sum((1, 2)).cpu().numpy()
    gj[2] = (g * hj).sum((0, 1)) / np.asarray(d["proportion"])
    scale, g_scale = max(1.0, np.abs(h_ref).max()), max(1.0, np.abs(grad_ref).max())
    for x in (h, hj):
        assert np.all(np.abs(x - h_ref) <= H_RTOL * np.abs(h_ref) + H_ATOL * scale), np.abs(x - h_ref).max()
    for x in (grad, gj):
        assert np.all(np.abs(x - grad_ref) <= G_RTOL * np.abs(grad_ref) + G_ATOL * g_scale), (x, grad_ref)
