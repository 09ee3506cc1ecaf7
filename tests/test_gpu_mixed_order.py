"""The FP32 predictor with rows on both sides of the length up to which its threads
take the particles as they are numbered, for ids along the lattice, against it and
shuffled: within 1e-5 of the FP64 predictor's largest velocity and dt times that in
the positions (the bound of the other tests of this predictor)."""
import numpy as np
import pytest

import voxarmps_amd as vx

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dim,re", [(2, 2.1), (2, 3.8), (2, 4.0), (3, 2.1), (3, 2.2), (3, 2.3)], ids=str)
@pytest.mark.parametrize("n", [70, 20011])
@pytest.mark.parametrize("order", ["first", "last", "shuffled"])
def test_predictor_of_any_numbering(hip, dim, re, n, order):
    rng = np.random.default_rng(n)
    side = int(np.ceil(n ** (1 / dim)))
    k = np.arange(n)
    lat = np.stack([k % side, k // side % side, k // side ** 2][:dim], 1)
    lat = lat[:, ::-1] if order == "last" else lat[rng.permutation(n)] if order == "shuffled" else lat
    pos = lat + rng.uniform(-0.1, 0.1, (n, dim))
    z = np.zeros(n)
    v = rng.normal(0, 1, (3, n))
    case = vx.Case(dim, 1.0, pos[:, 0].copy(), pos[:, 1].copy(), pos[:, 2].copy() if dim == 3 else z, v[0], v[1],
                   v[2] if dim == 3 else z.copy(), z.copy(), np.ones(n, np.int32))
    p = vx.default_params(dim, 1.0)
    p.re_s = p.re_l = re
    p.lambda_ = 0.16832 * re ** 2
    p.dt = 1e-3
    vx.set_box(p, case)
    out = []
    for precision in (vx._abi.PREC_FP64, vx._abi.PREC_MIXED):
        q = p.copy()
        q.precision = precision
        s = vx.Simulation(q, case, backend=hip)
        s.init()
        s.set("PHAT", np.linspace(0.0, 1.0, n))
        for st in ("PNUM", "VISCOSITY", "PREDICTION"):
            getattr(s, st)()
        out.append({f: s.get(f) for f in ("USTAR", "VSTAR", "WSTAR", "XSTAR", "YSTAR", "ZSTAR")})
        s.close()
    a, b = out
    top = max(np.abs(a[f]).max() for f in ("USTAR", "VSTAR", "WSTAR"))
    for f in ("USTAR", "VSTAR", "WSTAR")[:dim]:
        assert np.abs(a[f] - b[f]).max() <= 1e-5 * top, f
    for f in ("XSTAR", "YSTAR", "ZSTAR")[:dim]:
        assert np.abs(a[f] - b[f]).max() <= p.dt * 1e-5 * top + 2 ** -24 * side, f
