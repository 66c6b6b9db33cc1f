"""Blocked Gauss-Jordan inverse (21..128 DOF) against LAPACK: panel remainders, tile edges, rows that
need exchanging, equal candidates and a singular block among regular ones."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("sizes", [(21, 22, 23, 32), (33, 47, 48, 63, 64), (65, 97, 100, 111, 112), (113, 126, 127, 128)])
def test_blocked_inverse(sizes):
    import torch
    from scipy.linalg import lu_factor
    from bosss_amd.blocks import BlockBatch
    print("case block inverse", sizes, flush=True)
    rng = np.random.default_rng(2)
    mats = []
    for n in sizes:
        A = rng.uniform(-1, 1, (n, n))
        mats += [A, np.eye(n)[rng.permutation(n)] + 0.01 * A]           # exchanges in most and in all columns
        T = np.ones((n, n))
        T[np.tril_indices(n, -1)] = -1.0                                  # equal candidates in every column: no exchange
        mats.append(T)
        S = A.copy()
        S[:, n // 2] = 0.0
        mats.append(S)                                                     # singular: LU factors and INFO
    bb = BlockBatch([len(m) for m in mats])
    A = torch.from_numpy(np.concatenate([m.ravel() for m in mats])).to("cuda:0")
    ipiv = torch.zeros(bb.ndof, dtype=torch.int32, device="cuda:0")
    info = torch.full((bb.nblk,), 7, dtype=torch.int32, device="cuda:0")
    bb.factor(A, ipiv, info, inverse=True)
    A, ipiv, info = A.cpu().numpy(), ipiv.cpu().numpy(), info.cpu().numpy()
    for b, m in enumerate(mats):
        n, o, x = len(m), bb.off[b], bb.xoff[b]
        got, piv = A[o:o + n * n].reshape(n, n), ipiv[x:x + n] - 1
        if b % 4 == 3:
            lu, ref = lu_factor(m, check_finite=False)
            assert info[b] == n // 2 + 1
            assert np.abs(got - lu).max() < 1e-12 * n
        else:
            lu, ref = lu_factor(m)
            assert info[b] == 0
            inv = np.linalg.inv(m)
            # forward error of a backward stable inverse: n eps cond, one digit above
            assert np.abs(got - inv).max() <= 10 * n * 2.2e-16 * np.linalg.cond(m) * np.abs(inv).max()
        assert (piv == ref).all()
