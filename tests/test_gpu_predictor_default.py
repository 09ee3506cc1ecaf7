"""The predictor a context starts with on both sides of each line of its rule (particle
counts, dimension, row lengths): the variant, and the bits of the other variants."""
import numpy as np
import pytest

import voxarmps_amd as vx

pytestmark = pytest.mark.gpu

CASES = [(2, 49152, 2.1, 2.1, 8), (2, 49153, 2.1, 2.1, 7), (2, 65536, 2.1, 3.1, 8), (2, 65537, 2.1, 3.1, 7),
         (2, 98304, 2.1, 4.0, 8), (2, 98305, 2.1, 4.0, 7), (2, 131072, 4.0, 4.0, 8), (2, 131073, 4.0, 4.0, 7),
         (3, 98304, 2.1, 2.1, 8), (3, 98305, 2.1, 2.1, 6), (3, 98305, 2.1, 3.1, 8), (2, 1, 2.1, 4.0, 8)]


@pytest.mark.parametrize("dim,n,rs,rl,want", CASES, ids=str)
def test_default_predictor(hip, dim, n, rs, rl, want):
    rng = np.random.default_rng(n)
    side = int(np.ceil(n ** (1 / dim)))
    k = np.arange(n)
    pos = [q + rng.uniform(-0.1, 0.1, n) for q in (k % side, k // side % side, k // side ** 2)[:dim]]
    z = np.zeros(n)
    v = rng.normal(0, 1, (3, n))
    t = np.ones(n, np.int32)
    t[n // 2:] = 2
    case = vx.Case(dim, 1.0, pos[0], pos[1], pos[2] if dim == 3 else z, v[0], v[1],
                   v[2] if dim == 3 else z.copy(), z.copy(), t)
    p = vx.default_params(dim, 1.0)
    p.re_s, p.re_l = rs, rl
    p.lambda_ = 0.16832 * rl ** 2
    p.dt = 1e-3
    vx.set_box(p, case)
    s = vx.Simulation(p, case, backend=hip)
    assert s.tuning() == (0, 0, want, 0)
    s.init()
    for st in ("PNUM", "VISCOSITY"):
        getattr(s, st)()
    s.set("PHAT", rng.normal(0, 1, n))
    ref = None
    for variant in (want, 8, 6, 0):
        s.set_tuning([0, 0, variant, 0])
        s.PREDICTION()
        out = [s.get(f) for f in ("XSTAR", "YSTAR", "USTAR", "VSTAR") + (("ZSTAR", "WSTAR") if dim == 3 else ())]
        ref = ref or out
        for a, b in zip(out, ref):
            assert np.array_equal(a, b, equal_nan=True), variant
    s.close()
