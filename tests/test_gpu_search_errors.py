"""A neighbour search that ends on an error between counting the cells and placing
the particles leaves nothing behind: the next search's cells, lists and pressure
system are the oracle's. The error is one that an earlier call of the same thread
left in the HIP runtime (an allocation no device has room for), which the launch
check after the count reports."""
import ctypes as C

import numpy as np
import pytest

import voxarmps_amd as vx
from helpers import HipMem

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dim,n,ks,kl", [(2, 5000, 2.1, 3.1), (2, 60000, 2.1, 3.1), (3, 60000, 2.1, 3.1)], ids=str)
def test_search_after_an_unfinished_one(hip, oracle, dim, n, ks, kl):
    rng = np.random.default_rng(n + dim)
    side = int(np.ceil(n ** (1 / dim)))
    k = np.arange(n)
    pos = [q + rng.uniform(-0.2, 0.2, n) for q in (k % side, k // side % side, k // side ** 2)[:dim]]
    z = np.zeros(n)
    case = vx.Case(dim, 1.0, pos[0], pos[1], pos[2] if dim == 3 else z, z.copy(), z.copy(), z.copy(), z.copy(),
                   np.ones(n, np.int32))
    p = vx.default_params(dim, 1.0)
    p.re_s, p.re_l = ks, kl
    p.lambda_ = 0.16832 * p.re_l ** 2
    vx.set_box(p, case)
    sims = [vx.Simulation(p, case, backend=b) for b in (hip, oracle)]
    for s in sims:
        s.init()
    g, c = sims
    rt = HipMem(hip).rt
    for repeat in range(2):
        ptr = C.c_void_p()
        assert rt.hipMalloc(C.byref(ptr), C.c_size_t(1 << 60)) != 0
        with pytest.raises(vx.VoxError) as e:
            g.autotune(reps=1)
        assert e.value.code == vx._abi.VOX_ERR_HIP
        g.set_tuning([0, 0, 8, 0])
        for s in sims:
            for f in "XYZ"[:dim]:
                s.set(f, s.get(f) + 0.05 * np.sin(np.arange(n) + repeat))
            for st in ("PNUM", "NEIGHBOR"):
                getattr(s, st)()
        for w in (vx.LIST_S, vx.LIST_L):
            assert np.array_equal(g.cells(w), c.cells(w))
            for a, b in zip(g.neighbors(w), c.neighbors(w)):
                assert np.array_equal(a, b)
    for s in sims:
        s.NEIGHBOR()
        for st in ("VISCOSITY", "PREDICTION", "PNUMSTAR", "BCON", "MATRIX"):
            getattr(s, st)()
    a, b = g.ppe(), c.ppe()
    for key in ("ids", "rowptr", "cols", "vals", "rhs"):
        assert np.array_equal(a[key], b[key]), key
    for s in sims:
        s.close()
