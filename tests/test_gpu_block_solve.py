"""Solves with given factors (bosss_hip_block_solve, device and host arrays) at sizes around the limits of its
kernels: 64 and 128 DOF (registers), 4096 DOF (the vector in LDS) and above it, in one batch."""
import ctypes

import numpy as np
import pytest
import scipy.linalg as sla

pytestmark = pytest.mark.gpu

SIZES = [4101, 1, 64, 4096, 65, 128, 129, 4097]


def factors(n, rng):
    """Unit lower and upper factor of a well-conditioned system, and 1-based row exchanges."""
    lu = rng.uniform(-1, 1, (n, n)) / n
    lu[np.arange(n), np.arange(n)] = rng.uniform(1, 2, n)
    piv = np.arange(n)
    for j in rng.integers(0, n, n // 8 + 1):
        piv[j] = rng.integers(j, n)
    return lu, piv


@pytest.mark.parametrize("entry", ["bosss_hip_block_solve_dev", "bosss_hip_block_solve"])
def test_solve_at_the_limits_of_the_kernels(entry):
    import torch
    from bosss_amd._lib import lib
    from bosss_amd.operator import Context
    rng = np.random.default_rng(8)
    blocks = [factors(n, rng) for n in SIZES]
    n = np.array(SIZES, np.int32)
    n64 = n.astype(np.int64)
    off, xoff = np.cumsum(n64 ** 2) - n64 ** 2, np.cumsum(n64) - n64
    arrays = [n, off, np.concatenate([lu.ravel() for lu, _ in blocks]), np.concatenate([p + 1 for _, p in blocks]).astype(np.int32), xoff, xoff]
    x0 = rng.uniform(-1, 1, int(n64.sum()))
    print("case", entry, SIZES, flush=True)
    L, ctx, x = lib(), Context.get(0).h, x0.copy()
    if entry.endswith("_dev"):
        t = [torch.from_numpy(a).cuda() for a in arrays + [x]]
        p = [ctypes.c_void_p(a.data_ptr()) for a in t]
        rc = L.bosss_hip_block_solve_dev(ctx, len(n), *p, ctypes.c_void_p(torch.cuda.current_stream().cuda_stream))
        x = t[-1].cpu().numpy()
    else:
        fn = L.bosss_hip_block_solve
        rc = fn(ctx, len(n), *[a.ctypes.data_as(ty) for a, ty in zip(arrays + [x], fn.argtypes[2:])])
    assert rc == 0, L.bosss_hip_block_last_error().decode()
    for k, (lu, piv) in enumerate(blocks):
        s = slice(xoff[k], xoff[k] + n64[k])
        want = sla.lu_solve((lu, piv), x0[s], check_finite=False)
        # substitution error: n rounding steps on rows of |L|, |U| with sums below 2, n eps |x| each way
        assert np.abs(x[s] - want).max() <= 4 * max(n64[k], 8) * 2.3e-16 * np.abs(want).max(), (SIZES[k], np.abs(x[s] - want).max())
