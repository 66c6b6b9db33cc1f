"""Direct assembly of the linear forms (SIP, upwind + SIP): every compiled degree, on graded grids
with boundary and periodic directions, against the oracle's exact Jacobian blocks."""
import sys

import numpy as np
import pytest

from oracle.bosss_ref import RefModel, params_vector, OP_SIP, OP_ADVDIFF

pytestmark = pytest.mark.gpu
KIND = {"sip": OP_SIP, "advdiff": OP_ADVDIFF}


@pytest.mark.parametrize("form,p,shape,per", [
    ("sip", 1, (3, 4), (False, True)), ("sip", 2, (7, 5), (False, False)), ("sip", 3, (1, 3), (False, False)),
    ("sip", 1, (3, 3, 4), (True, False, False)), ("sip", 2, (1, 1, 2), (False, False, False)), ("sip", 3, (3, 4, 3), (True, True, True)),
    ("advdiff", 2, (9, 8), (True, False)), ("advdiff", 2, (4, 3, 5), (False, True, False)), ("advdiff", 3, (5, 3, 3), (False, False, True))])
def test_direct_assembly_matches_oracle_blocks(form, p, shape, per):
    import torch
    from bosss_amd.grid import CartesianGrid
    from bosss_amd.operator import DifferentialOperator, default_quad_order
    print("case direct assembly", form, p, shape, per, flush=True)
    sys.stdout.flush()
    D = len(shape)
    rng = np.random.default_rng(5)
    nodes = [np.concatenate([[0.0], np.cumsum(rng.uniform(0.5, 1.5, n))]) for n in shape]
    g = CartesianGrid(nodes=nodes, periodic=per)
    nu, vel = (1.0 if form == "sip" else -0.01), (1.0, -0.5, 0.25)[:D]
    ref = RefModel(D, shape, p, default_quad_order(form, p), periodic=[int(x) for x in per], nodes=nodes)
    diag, offd = ref.assemble(KIND[form], params_vector(1.3, nu, vel + (0.0,) * (3 - D)))
    op = DifferentialOperator(g, form, p, nu=nu, velocity=vel)
    ev = op.GetMatrixBuilder()
    N, S = op.N, ev.S
    want = np.zeros((g.J, S, N, N))
    want[:, 0] = diag
    for e in range(g.E):
        ci, co = g.cells[e]
        if co >= 0:
            want[ci, 1 + g.trafo[e, 0]] = offd[e, 0]
            want[co, 1 + g.trafo[e, 1]] = offd[e, 1]
    scale = np.abs(diag).max()
    U = torch.zeros(op.ndof, dtype=torch.float64, device="cuda:0")
    B = torch.full((ev.entries,), float("nan"), dtype=torch.float64, device="cuda:0")
    op.assemble_dev(U, B)                                   # beta = 0 overwrites every entry
    got = B.cpu().numpy().reshape(g.J, S, N, N)
    assert np.abs(got - want).max() < 1e-12 * scale
    op.assemble_dev(U, B, alpha=-2.0, beta=0.5)             # blocks <- 0.5 old - 2 new
    assert np.abs(B.cpu().numpy().reshape(got.shape) + 1.5 * want).max() < 1e-12 * scale
    d = torch.full((g.J * N * N,), float("nan"), dtype=torch.float64, device="cuda:0")
    for transposed in (False, True):
        op.diag_blocks_dev(U, d, alpha=0.7, shift=3.0, transposed=transposed)
        blk = d.cpu().numpy().reshape(g.J, N, N)
        blk = blk.transpose(0, 2, 1) if transposed else blk
        assert np.abs(blk - 0.7 * diag - 3.0 * np.eye(N)).max() < 1e-12 * scale
