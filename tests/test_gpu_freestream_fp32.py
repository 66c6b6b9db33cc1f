"""FP32 Euler residual of constant states: volume and face terms of a cell cancel, cell by cell up to rounding, and on
average over many states up to what the rounded tables leave."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("form", ["euler_lf", "euler_hllc"])
def test_volume_and_faces_agree_on_average(form, monkeypatch):
    import torch
    from bosss_amd.grid import CartesianGrid
    from bosss_amd.operator import DifferentialOperator
    print("case free stream fp32", form, flush=True)
    monkeypatch.setenv("BOSSS_HIP_SPLIT", "0")
    J, p, rng = 16384, 3, np.random.default_rng(0)
    # one cell in y and z, its own neighbour: the residual of a mode that varies in y (or z) alone is volume minus faces
    h = [1 / 8, 0.137, 0.211]
    g = CartesianGrid(nodes=[np.arange(J + 1.0) * h[0], np.array([0, h[1]]), np.array([0, h[2]])], periodic=[True] * 3)
    op = DifferentialOperator(g, form, p, gamma=1.4, precision="fp32")
    rho, vel, pr = rng.uniform(0.5, 1.5, J), rng.uniform(0.5, 1.5, (J, 3)), rng.uniform(0.5, 1.5, J)
    E = pr / 0.4 + 0.5 * rho * (vel ** 2).sum(1)
    U = np.zeros((J, 5, op.N))
    U[:, :, 0] = np.concatenate([rho[:, None], rho[:, None] * vel, E[:, None]], 1) * np.sqrt(np.prod(h))
    Ut = torch.from_numpy(U.reshape(-1)).to("cuda:0", torch.float32)
    R = torch.empty_like(Ut)
    op.evaluate_dev(Ut, R)
    R = R.double().cpu().numpy().reshape(J, 5, op.N)
    modes = [(a, b, d - a - b) for d in range(p + 1) for a in range(d + 1) for b in range(d - a + 1)]
    for d in (1, 2):
        F = np.stack([rho * vel[:, d]] + [rho * vel[:, d] * vel[:, i] + (pr if i == d else 0.0) for i in range(3)] + [(E + pr) * vel[:, d]], 1)
        for a in (1, 3):
            m = modes.index(tuple(a if i == d else 0 for i in range(3)))
            face = 2 * h[0] * h[3 - d] * np.sqrt((2 * a + 1) / np.prod(h)) * F     # what the two faces contribute
            share = (face * R[:, :, m]).sum() / (face ** 2).sum()
            rms = np.sqrt((R[:, :, m] ** 2).mean() / (face ** 2).mean())
            print("  direction %d, degree %d: %.1e on average, %.1e per cell" % (d, a, share, rms), flush=True)
            # the derivative factor is carried in two floats, so what is left is the average of the weights' and
            # traces' roundings, below the 2^-24 of a single one; a cell adds those of its sums over 125 nodes
            assert abs(share) < 2.0 ** -24 and rms < 16 * 2.0 ** -24
