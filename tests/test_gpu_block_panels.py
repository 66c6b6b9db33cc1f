"""Blocks above 128 DOF at the edges of the register panels and of the solve's tiles: factors and
pivots against LAPACK, residual of the solve, zero pivots, with and without pivots asked for."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("sizes", [(129, 128, 160, 161, 1), (255, 256, 257, 64), (512, 513, 191, 193), (1023, 1024, 31), (1025, 200)])
def test_register_panels(sizes):
    import torch
    from scipy.linalg import lu_factor
    from bosss_amd.blocks import BlockBatch
    print("case block panels", sizes, flush=True)
    rng = np.random.default_rng(6)
    mats = [rng.uniform(-1, 1, (n, n)) for n in sizes]
    zero = rng.uniform(-1, 1, (sizes[0], sizes[0]))
    zero[:, sizes[0] - 40] = 0.0
    mats.append(zero)
    bb = BlockBatch([len(m) for m in mats])
    A0 = torch.from_numpy(np.concatenate([m.ravel() for m in mats])).to("cuda:0")
    A, B = A0.clone(), A0.clone()
    ipiv = torch.zeros(bb.ndof, dtype=torch.int32, device="cuda:0")
    info, info2 = [torch.full((bb.nblk,), 7, dtype=torch.int32, device="cuda:0") for _ in range(2)]
    b = rng.uniform(-1, 1, bb.ndof)
    x = torch.from_numpy(b).to("cuda:0")
    bb.factor(A, ipiv, info)
    bb.factor(B, None, info2)              # no pivots kept: the forms with their own state
    bb.solve(A, ipiv, x)
    A, B, ipiv, x = A.cpu().numpy(), B.cpu().numpy(), ipiv.cpu().numpy(), x.cpu().numpy()
    assert info.tolist() == info2.tolist() == [0] * len(sizes) + [sizes[0] - 39]
    for k, m in enumerate(mats):
        n, o, r = len(m), bb.off[k], bb.xoff[k]
        lu, piv = lu_factor(m, check_finite=False) if k < len(sizes) else (None, None)
        F = A[o:o + n * n].reshape(n, n)
        assert np.abs(F - B[o:o + n * n].reshape(n, n)).max() < 1e-10 * np.abs(F).max()
        if lu is None:
            continue
        assert (ipiv[r:r + n] - 1 == piv).all()
        L, U = np.tril(F, -1) + np.eye(n), np.triu(F)
        P = m.copy()
        for j, q in enumerate(piv):
            P[[j, q]] = P[[q, j]]
        assert np.abs(L @ U - P).max() < 2.2e-16 * n * np.abs(U).max()          # backward error of partial pivoting
        xs = x[r:r + n]
        assert np.abs(m @ xs - b[r:r + n]).max() < 2.2e-16 * n * np.abs(U).max() * n * np.abs(xs).max()
