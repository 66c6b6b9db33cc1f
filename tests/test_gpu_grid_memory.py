"""What a grid holds on the device, and operators that share one grid."""
import ctypes
import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def test_euler_grid_holds_the_uploaded_metrics_alone():
    import torch
    from bosss_amd.grid import CartesianGrid
    from bosss_amd.operator import DifferentialOperator
    print("case grid memory", flush=True)
    DifferentialOperator(CartesianGrid((2, 2, 2), periodic=[True] * 3), "euler_hllc", 3)   # modules loaded
    g = CartesianGrid((80, 80, 80), periodic=[True] * 3)
    torch.cuda.synchronize()
    free0 = torch.cuda.mem_get_info(0)[0]
    op = DifferentialOperator(g, "euler_hllc", 3)
    torch.cuda.synchronize()
    held = free0 - torch.cuda.mem_get_info(0)[0]
    # detJ, scaling, lenscale (1 double each), invJ (9), sqrtg (6), normals (18), neighbours (6 ints); every
    # array and table in an allocation of its own, rounded up to 2 MiB
    metrics = g.J * (8 * (3 + 9 + 6 + 18) + 4 * 6)
    assert held <= metrics + 12 * (2 << 20), (held, metrics)
    op.close()


def test_operators_of_one_grid_made_by_threads():
    import torch
    from bosss_amd import _lib
    from bosss_amd.grid import CartesianGrid
    from bosss_amd.operator import FORMS, DifferentialOperator
    print("case shared grid", flush=True)
    g = CartesianGrid((9, 7, 5), periodic=[True] * 3)
    euler = DifferentialOperator(g, "euler_lf", 2)            # its grid has no cell-fastest metrics yet
    alone = DifferentialOperator(g, "sip", 2)
    t = alone.tables
    keep = [np.ascontiguousarray(x) for x in (t.vw, t.phi, t.dphi, t.fw, t.trace, t.dtrace)]
    dp = lambda a: a.ctypes.data_as(ctypes.POINTER(ctypes.c_double))
    td = _lib.TablesDesc(3, 2, t.N, t.Kv, t.Ke, t.ntrafo, *[dp(x) for x in keep])
    fp = _lib.FormParams(1.3, 1.0, (ctypes.c_double * 3)(), 1.4, 1.0)
    hs, rcs = [ctypes.c_void_p() for _ in range(4)], [None] * 4

    def make(i):
        rcs[i] = _lib.lib().bosss_hip_op_create(euler.ctx.h, euler._grid_h, ctypes.byref(td), FORMS["sip"], ctypes.byref(fp), 0, ctypes.byref(hs[i]))

    threads = [threading.Thread(target=make, args=(i,)) for i in range(4)]
    [x.start() for x in threads]
    [x.join() for x in threads]
    assert rcs == [0] * 4
    U = torch.from_numpy(np.random.default_rng(0).uniform(-1, 1, alone.ndof)).cuda()
    want, got = torch.empty_like(U), torch.empty_like(U)
    alone.evaluate_dev(U, want)
    for h in hs:
        got.fill_(float("nan"))
        _lib.check(_lib.lib().bosss_hip_evaluate_dev(h, 1.0, 0.0, U.data_ptr(), got.data_ptr(), torch.cuda.current_stream().cuda_stream))
        assert torch.equal(got, want)
        _lib.lib().bosss_hip_op_destroy(h)
