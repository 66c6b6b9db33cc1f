"""Modal kernels of the linear scalar forms (axis-aligned cells) against the nodal tensor-table
kernels: the same grid rotated as a whole, cells, normals and transport velocity, has the same
residual, and its cells are not axis-aligned any more, so it takes the nodal kernels."""
import sys

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def rotation(D):
    c, s = np.cos(0.4), np.sin(0.4)
    if D == 2:
        return np.array([[c, -s], [s, c]])
    a, b = np.array([[c, -s, 0], [s, c, 0], [0, 0, 1.0]]), np.array([[1.0, 0, 0], [0, c, -s], [0, s, c]])
    return a @ b


@pytest.mark.parametrize("form,p,shape,per,prec", [
    ("sip", 1, (9, 5), (False, True), "fp64"), ("sip", 2, (8, 8), (False, False), "fp64"), ("sip", 3, (13, 11), (True, False), "fp64"),
    ("sip", 1, (5, 3, 5), (False, True, False), "fp64"), ("sip", 2, (1, 1, 1), (False, False, False), "fp64"),
    ("sip", 3, (4, 2, 8), (True, True, True), "fp64"), ("advdiff", 2, (7, 10), (True, False), "fp64"),
    ("advdiff", 2, (3, 5, 5), (False, False, True), "fp64"), ("advdiff", 3, (5, 4, 7), (False, True, False), "fp64"),
    ("advdiff", 3, (2, 1, 3), (True, True, True), "fp64"), ("advdiff", 3, (5, 4, 7), (False, True, False), "fp32")])
def test_modal_kernels_equal_nodal_kernels(form, p, shape, per, prec):
    import torch
    from bosss_amd.grid import CartesianGrid
    from bosss_amd.operator import DifferentialOperator
    print("case modal", form, p, shape, per, prec, flush=True)
    sys.stdout.flush()
    D = len(shape)
    rng = np.random.default_rng(8)
    nodes = [np.concatenate([[0.0], np.cumsum(rng.uniform(0.5, 1.5, n))]) for n in shape]
    Q = rotation(D)
    vel = np.array((0.7, -0.5, 0.25)[:D])
    ops = []
    for rot in (False, True):
        g = CartesianGrid(nodes=nodes, periodic=per)
        if rot:
            g.invJ = g.invJ @ Q.T           # xi = invJ Q^T x'
            g.normals = g.normals @ Q.T
        ops.append(DifferentialOperator(g, form, p, nu=1.0 if form == "sip" else -0.3, velocity=tuple(Q @ vel if rot else vel), precision=prec))
        assert ops[-1].uses_tensor_tables()
    dt = torch.float64 if prec == "fp64" else torch.float32
    tol = 1e-12 if prec == "fp64" else 2e-5
    U, W, R0 = [torch.from_numpy(rng.uniform(-1, 1, ops[0].ndof)).to("cuda:0", dt) for _ in range(3)]
    res = []
    for op in ops:
        out = []
        R = torch.full_like(U, float("nan"))
        op.evaluate_dev(U, R)               # beta = 0 overwrites every entry
        out.append(R)
        R = R0.clone()
        op.evaluate_dev(U, R, alpha=-1.5, beta=0.5)
        out.append(R)
        for call in (op.jvp_dev, op.vjp_dev):
            y = torch.full_like(U, float("nan"))
            call(U, W, y)
            out.append(y)
        R, y = R0.clone(), torch.full_like(U, float("nan"))
        op.evaluate_vjp_dev(U, R, W, y, alpha=2.0, beta=1.0)
        res.append([t.double().cpu().numpy() for t in out + [R, y]])
    for k, (a, b) in enumerate(zip(*res)):
        assert np.abs(a - b).max() < tol * np.abs(b).max(), k
    # the adjoint is the transpose of the JVP
    a, b = float(np.dot(res[0][2], R0.double().cpu().numpy())), torch.empty_like(U)
    ops[0].vjp_dev(U, R0, b)
    b = float(torch.dot(b.double(), W.double()))
    assert abs(a - b) < tol * np.abs(res[0][2]).sum()
