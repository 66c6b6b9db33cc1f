"""Diagonal blocks of the Euler Jacobian from moments, against own-cell JVP probes on the general
quadrature tables (an operator created with BOSSS_HIP_GENERIC_TABLES=1)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("form,p,shape", [
    ("euler_hllc", 2, (1, 1, 1)), ("euler_hllc", 2, (3, 1, 2)), ("euler_lf", 2, (3, 4, 5)),
    ("euler_hllc", 3, (1, 2, 3)), ("euler_lf", 3, (2, 3, 3)), ("euler_hllc", 3, (9, 11, 7))])
def test_moment_blocks_equal_probes(form, p, shape, monkeypatch):
    import torch
    from bosss_amd.grid import CartesianGrid
    from bosss_amd.operator import DifferentialOperator
    print("case euler blocks", form, p, shape, flush=True)
    D = len(shape)
    rng = np.random.default_rng(4)
    g = CartesianGrid(nodes=[np.concatenate([[0.0], np.cumsum(rng.uniform(0.5, 1.5, n))]) for n in shape], periodic=[True] * D)
    if form == "euler_lf":      # cells, normals and all, rotated: a full inverse Jacobian
        c, t = np.cos(0.4), np.sin(0.4)
        Q = np.array([[c, -t, 0], [t, c, 0], [0, 0, 1.0]]) @ np.array([[1.0, 0, 0], [0, c, -t], [0, t, c]])
        g.invJ, g.normals = g.invJ @ Q.T, g.normals @ Q.T
    op = DifferentialOperator(g, form, p, gamma=1.4)
    assert op.uses_tensor_tables()
    monkeypatch.setenv("BOSSS_HIP_GENERIC_TABLES", "1")
    probe = DifferentialOperator(g, form, p, gamma=1.4)
    assert not probe.uses_tensor_tables()
    monkeypatch.delenv("BOSSS_HIP_GENERIC_TABLES")
    V, N = op.nvars, op.N
    s0 = np.sqrt(g.detJ * 2.0 ** D)[:, None]
    rho, vel, pr = rng.uniform(0.8, 1.2, g.J), rng.uniform(-1.4, 1.4, (g.J, D)), rng.uniform(0.9, 1.1, g.J)   # sub- and supersonic
    mean = np.concatenate([rho[:, None], rho[:, None] * vel, (pr / 0.4 + 0.5 * rho * (vel ** 2).sum(1))[:, None]], 1) * s0
    U = 0.02 * rng.uniform(-1, 1, (g.J, V, N)) * s0[:, :, None]
    U[:, :, 0] = mean
    U = torch.from_numpy(U.reshape(-1)).float().double().to("cuda:0")
    NT = V * N
    for alpha, shift, transposed in ((1.0, 0.0, False), (0.7, 3.0, True)):
        A, B = [torch.full((g.J * NT * NT,), float("nan"), dtype=torch.float64, device="cuda:0") for _ in range(2)]
        op.diag_blocks_dev(U, A, alpha=alpha, shift=shift, transposed=transposed)
        probe.diag_blocks_dev(U, B, alpha=alpha, shift=shift, transposed=transposed)
        scale = float(B.abs().max())
        assert float((A - B).abs().max()) < 1e-12 * scale
        # an FP32 operator evaluates its FP32 state in 64 bits
        C = torch.full_like(A, float("nan"))
        DifferentialOperator(g, form, p, gamma=1.4, precision="fp32").diag_blocks_dev(U.float(), C, alpha=alpha, shift=shift,
                                                                                       transposed=transposed)
        assert float((A - C).abs().max()) == 0.0
