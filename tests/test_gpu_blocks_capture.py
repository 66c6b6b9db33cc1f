"""Matrix and diagonal blocks captured into a graph by an operator that has made its staging vectors (a host call) but
no blocks yet: replays equal the eager call, before and after it has made the tables of the direct forms."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("form,p,shape", [("sip", 2, (3, 4, 5)), ("advdiff", 3, (4, 3, 3)), ("advdiff", 2, (5, 4)),
                                          ("euler_hllc", 2, (3, 3, 4)), ("euler_lf", 2, (4, 5))])
def test_blocks_captured_before_their_first_call(form, p, shape):
    import torch
    from bosss_amd.grid import CartesianGrid
    from bosss_amd.operator import DifferentialOperator
    from bosss_amd.workloads import euler_state
    print("case blocks under capture", form, p, shape, flush=True)
    euler, D = form.startswith("euler"), len(shape)
    kw = {} if euler else dict(nu=-0.3, velocity=(1.0, 0.5, 0.25))
    op = DifferentialOperator(CartesianGrid(shape, periodic=[euler] * D), form, p, **kw)
    states = [euler_state(op.grid, op.N, seed=s, perturb=0.02) if euler else np.random.default_rng(s).uniform(-1, 1, op.ndof) for s in range(3)]
    op.evaluate(states[0])                    # host call: staging vectors
    _, entries, _, _ = op.matrix_layout()
    nd = op.grid.J * (op.nvars * op.N) ** 2
    U = torch.from_numpy(states[0]).cuda()
    new = lambda n: torch.zeros(n, dtype=torch.float64, device="cuda:0")

    def capture():
        diag, mat, graph = new(nd), None if euler else new(entries), torch.cuda.CUDAGraph()
        torch.cuda.synchronize()
        with torch.cuda.graph(graph):
            op.diag_blocks_dev(U, diag, alpha=0.7, shift=2.0, transposed=True)
            if mat is not None:
                op.assemble_dev(U, mat, alpha=0.7)
        return graph, diag, mat

    def check(graph, diag, mat):
        for s in states:
            U.copy_(torch.from_numpy(s))
            diag.fill_(float("nan"))
            graph.replay()
            torch.cuda.synchronize()
            wd, wm = new(nd), new(entries)
            op.diag_blocks_dev(U, wd, alpha=0.7, shift=2.0, transposed=True)
            # the forms differ in rounding alone: sums of at most 6 faces and 125 nodes
            assert float((diag - wd).abs().max()) < 1e-12 * float(wd.abs().max())
            if mat is not None:
                op.assemble_dev(U, wm, alpha=0.7)
                assert float((mat - wm).abs().max()) < 1e-12 * float(wm.abs().max())

    first = capture()
    check(*first)
    check(*capture())
    check(*first)
