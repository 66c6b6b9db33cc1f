"""Every form that factors blocks above 128 DOF, by what selects it: register panels (pivots kept, up to 1024 DOF), one
workgroup per block (no pivots kept), two launches per panel (no pivots kept and large blocks, or above 1024 DOF; with
allocated state words, or the fixed ones of the call that does not allocate).  Each call holds a zero column, a zero diagonal
with a pivot below, tied pivot candidates and a NaN, and follows another of other sizes whose state words it must not see."""
import ctypes

import numpy as np
import pytest

from oracle.bosss_ref import ref_block_lu

pytestmark = pytest.mark.gpu

MID, LARGE, HUGE = [150, 140, 129, 160], [520, 150, 513, 600], [1100, 129, 140, 1030]
COL = 36


def batch(sizes, seed):
    rng = np.random.default_rng(seed)
    blocks = [rng.uniform(-1, 1, (n, n)) + 0.2 * n * np.eye(n) for n in sizes]
    blocks[0][:, COL] = 0.0                                 # zero pivot: INFO = COL + 1, factorisation goes on
    blocks[1][:, :COL] = 0.0                                # unit columns, then a zero diagonal entry
    blocks[1][:COL, :COL] = np.eye(COL)
    blocks[1][COL, COL] = 0.0
    n = sizes[2]                                            # candidates of equal size: the first row wins
    blocks[2][:, 0] = np.where(np.arange(n) % 3 == 1, 4.0, -4.0)
    blocks[3][4, 0] = np.nan
    return blocks


@pytest.mark.parametrize("entry,pivots,calls", [
    ("bosss_hip_block_lu_dev", True, [LARGE, MID]), ("bosss_hip_block_lu_dev", False, [MID, LARGE, MID]),
    ("bosss_hip_block_lu_dev", True, [HUGE, HUGE[::-1]]), ("bosss_hip_block_lu_noalloc_dev", True, [HUGE, MID]),
    ("bosss_hip_block_lu_noalloc_dev", False, [LARGE, MID, HUGE])])
def test_factors_of_every_form(entry, pivots, calls):
    import torch
    from bosss_amd._lib import lib
    from bosss_amd.operator import Context
    L = lib()
    p = lambda t: ctypes.c_void_p(t.data_ptr()) if t is not None else None
    for i, sizes in enumerate(calls):
        print("case", entry, "pivots" if pivots else "no pivots", sizes, flush=True)
        blocks = batch(sizes, 17 + i)
        LUref, pivref, inforef, off, poff = ref_block_lu(sizes, blocks)
        assert list(inforef) == [COL + 1, 0, 0, 0] and pivref[poff[1] + COL] != COL and pivref[poff[2]] == 0 and pivref[poff[3] + 4] == 4
        n_t, off_t, poff_t = [torch.from_numpy(np.asarray(a)).cuda() for a in (np.array(sizes, np.int32), off, poff)]
        A = torch.from_numpy(np.concatenate([b.ravel() for b in blocks])).cuda()
        ipiv = torch.zeros(sum(sizes), dtype=torch.int32, device="cuda:0") if pivots else None
        info = torch.full((len(sizes),), -7, dtype=torch.int32, device="cuda:0")
        rc = getattr(L, entry)(Context.get(0).h, len(sizes), max(sizes), p(n_t), p(off_t), p(A), p(ipiv), p(poff_t) if pivots else None, p(info), 0,
                               ctypes.c_void_p(torch.cuda.current_stream().cuda_stream))
        assert rc == 0, L.bosss_hip_block_last_error().decode()
        assert info.cpu().tolist() == list(inforef)
        if pivots:
            assert (ipiv.cpu().numpy() == pivref + 1).all()
        LU = A.cpu().numpy()
        for b, n in enumerate(sizes[:3]):
            s = slice(off[b], off[b] + n * n)
            assert np.abs(LU[s] - LUref[s]).max() < 1e-12 * np.abs(LUref[s]).max(), (b, n)
