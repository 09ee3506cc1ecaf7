"""The one-block and the two-launch scan around the tile (4096), the limit (16384)
and a single item: unknown numbering, cells and lists of clouds of those sizes are
the oracle's, on repeated searches (each scan clears the counts of the next)."""
import numpy as np
import pytest

import voxarmps_amd as vx

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 1023, 4095, 4096, 4097, 16383, 16384, 16385, 20481])
def test_scans_of_any_length(hip, oracle, n):
    rng = np.random.default_rng(n)
    side = int(np.ceil(np.sqrt(n)))
    k = rng.permutation(side * side)[:n]
    z = np.zeros(n)
    case = vx.Case(2, 1.0, k % side + rng.uniform(-0.2, 0.2, n), k // side + rng.uniform(-0.2, 0.2, n), z,
                   z.copy(), z.copy(), z.copy(), z.copy(), rng.choice(np.array([0, 1, 1], np.int32), n))
    p = vx.default_params(2, 1.0)
    p.re_s, p.re_l = 2.1, 3.1
    p.lambda_ = 0.16832 * p.re_l ** 2
    vx.set_box(p, case)
    sims = [vx.Simulation(p, case, backend=b) for b in (hip, oracle)]
    for s in sims:
        s.init()
        s.set_n0(6.0, 12.0)
        s.NEIGHBOR()
    for repeat in range(2):
        for w in (vx.LIST_S, vx.LIST_L):
            assert np.array_equal(sims[0].cells(w), sims[1].cells(w))
            for a, b in zip(sims[0].neighbors(w), sims[1].neighbors(w)):
                assert np.array_equal(a, b)
        if repeat:
            break
        for s in sims:
            for f in ("X", "Y"):
                s.set(f, s.get(f) + 0.3 * np.sin(np.arange(n)))
            for st in ("NEIGHBOR", "PNUM", "VISCOSITY", "PREDICTION", "PNUMSTAR", "BCON", "MATRIX"):
                getattr(s, st)()
        a, b = sims[0].ppe(), sims[1].ppe()
        for key in ("ids", "rowptr", "cols"):
            assert np.array_equal(a[key], b[key]), key
    for s in sims:
        s.close()
