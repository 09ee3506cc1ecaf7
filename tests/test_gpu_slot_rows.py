"""vox_cgm_slot's row sums at lengths around their batches (16 lanes, 4 slots a
lane), with what a row may hold beside its couplings: ids out of range, the row
itself, and Dirichlet neighbours whose coefficients are not finite - none of
them counts. Against a dense FP64 solve."""
import ctypes as C

import numpy as np
import pytest
import torch

import voxarmps_amd as vx

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("entry", ["vox_cgm_slot", "vox_cgm_slot_noalloc"])
@pytest.mark.parametrize("length", [0, 1, 14, 15, 16, 17, 62, 63, 64, 65, 127, 130])
def test_rows_of_any_length(hip, entry, length):
    rng = np.random.default_rng(length)
    tp, junk = 150, 5
    stride = 2 + (length + junk) * 2 + 1
    free = np.ones(tp + 1, bool)
    free[rng.choice(np.arange(1, tp + 1), 15, replace=False)] = False
    ids = [i for i in range(1, tp + 1) if free[i]]
    A = np.zeros((tp + 1, tp + 1))
    for n, i in enumerate(ids):                        # symmetric: pairs at cyclic distances
        for d in range(1, length // 2 + 1):
            j = ids[(n + d) % len(ids)]
            if j != i:
                A[i, j] = A[j, i] = -rng.uniform(0.1, 1.0)
    neighb = np.zeros((tp + 1, stride), np.int32)
    poiss = np.zeros((tp + 1, stride))
    walls = np.flatnonzero(~free)
    for i in range(1, tp + 1):
        cols = list(np.flatnonzero(A[i]))
        vals = [A[i, j] for j in cols]
        A[i, i] = 1.0 - A[i].sum()
        cols += [0, tp + 1, -3, i, int(walls[0]) if walls[0] else int(walls[1])]
        vals += [7.0, np.nan, np.inf, 3.0, np.inf]
        order = rng.permutation(len(cols))
        neighb[i, 1] = len(cols) + 1
        neighb[i, 2:2 + len(cols)] = np.array(cols)[order]
        poiss[i, 1] = A[i, i]
        poiss[i, 2:2 + len(cols)] = np.array(vals)[order]
    b = rng.normal(size=tp + 1)
    want = np.zeros(tp + 1)
    want[ids] = np.linalg.solve(A[np.ix_(ids, ids)], b[ids])
    dev = [torch.from_numpy(a).cuda() for a in
           (neighb, poiss, b, np.where(free, 0, 1).astype(np.int32))]
    x = torch.full((tp + 1,), 9.0, dtype=torch.float64, device="cuda")
    info = vx._abi.VoxSolveInfo()
    f = getattr(hip.lib, entry)
    f.restype = C.c_int
    rc = f(C.c_int(tp), C.c_int(stride), *(C.c_void_p(a.data_ptr()) for a in dev),
           C.c_void_p(x.data_ptr()), C.c_double(1e-12), C.c_int(500), C.byref(info))
    assert rc == 0 and info.converged
    got = x.cpu().numpy()
    assert np.linalg.norm(got[ids] - want[ids]) <= 1e-10 * np.linalg.norm(want[ids])
    assert not got[1:][~free[1:]].any()
