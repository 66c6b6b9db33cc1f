"""Cell-split forms of the Euler kernels (four wavefronts share 16 cells) against the forms with 16
cells per wavefront: every variant, cell counts around multiples of 16 and 64."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("form,p,shape,prec", [
    ("euler_hllc", 2, (1, 1), "fp64"), ("euler_lf", 2, (17, 5), "fp64"), ("euler_hllc", 2, (3, 5, 1), "fp64"),
    ("euler_lf", 2, (4, 4, 4), "fp32"), ("euler_hllc", 3, (1, 1, 1), "fp64"), ("euler_lf", 3, (13, 5, 1), "fp64"),
    ("euler_hllc", 3, (4, 4, 1), "fp32"), ("euler_hllc", 3, (7, 11, 9), "fp64")])
def test_split_kernels_equal_whole_kernels(form, p, shape, prec, monkeypatch):
    import torch
    from bosss_amd.grid import CartesianGrid
    from bosss_amd.operator import DifferentialOperator
    print("case split", form, p, shape, prec, flush=True)
    D = len(shape)
    rng = np.random.default_rng(12)
    g = CartesianGrid(nodes=[np.concatenate([[0.0], np.cumsum(rng.uniform(0.5, 1.5, n))]) for n in shape], periodic=[True] * D)
    s0 = np.sqrt(g.detJ * 2.0 ** D)[:, None]
    rho, vel, pr = rng.uniform(0.8, 1.2, g.J), rng.uniform(-0.1, 0.1, (g.J, D)), rng.uniform(0.9, 1.1, g.J)
    mean = np.concatenate([rho[:, None], rho[:, None] * vel, (pr / 0.4 + 0.5 * rho * (vel ** 2).sum(1))[:, None]], 1) * s0
    dt, tol = (torch.float64, 1e-12) if prec == "fp64" else (torch.float32, 2e-5)
    res = []
    for split in ("0", "1"):
        monkeypatch.setenv("BOSSS_HIP_SPLIT", split)
        op = DifferentialOperator(g, form, p, gamma=1.4, precision=prec)
        r = np.random.default_rng(5)
        U = 0.02 * r.uniform(-1, 1, (g.J, op.nvars, op.N)) * s0[:, :, None]
        U[:, :, 0] = mean
        U, W, R0 = [torch.from_numpy(x.reshape(-1)).to("cuda:0", dt) for x in (U, r.uniform(-1, 1, op.ndof), r.uniform(-1, 1, op.ndof))]
        out = [torch.full_like(U, float("nan")) for _ in range(4)] + [R0.clone(), R0.clone()]
        op.evaluate_dev(U, out[0])                     # beta = 0 overwrites every entry
        op.jvp_dev(U, W, out[1])
        op.vjp_dev(U, W, out[2])
        op.evaluate_vjp_dev(U, out[4], W, out[3], alpha=-1.5, beta=0.5)
        op.evaluate_dev(U, out[5], alpha=2.0, beta=1.0)
        res.append([x.double().cpu().numpy() for x in out])
    for k, (a, b) in enumerate(zip(*res)):
        assert np.abs(a - b).max() < tol * max(1.0, np.abs(a).max()), k
