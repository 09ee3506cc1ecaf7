"""The stages that give a particle 16 lanes in small systems and one thread in
large ones: both sides of the line, few particles, and rows of any length (a clump,
far stragglers), against the oracle bit for bit; the Herschel-Bulkley viscosity to
1e-13 (pow)."""
import numpy as np
import pytest

import voxarmps_amd as vx

pytestmark = pytest.mark.gpu


def _cloud(dim, n, kind):
    rng = np.random.default_rng(n + dim)
    if kind == "lattice":
        side = int(np.ceil(n ** (1 / dim)))
        k = np.arange(n)
        pos = np.stack([k % side, k // side % side, k // side ** 2][:dim], 1) + rng.uniform(-0.3, 0.3, (n, dim))
    else:
        pos = np.concatenate([rng.uniform(0, 0.9, (n // 3, dim)) + 3.0, rng.uniform(0, 8, (n // 3, dim)),
                              rng.uniform(0, 90, (n - 2 * (n // 3), dim))])
    z = np.zeros(n)
    v = rng.normal(0, 1, (3, n))
    t = rng.choice(np.array([-1, 0, 1, 1, 2], np.int32), n)
    t = np.sort(t, kind="stable")                      # dummies, walls, fluid: the library's order
    return vx.Case(dim, 1.0, pos[:, 0].copy(), pos[:, 1].copy(), pos[:, 2].copy() if dim == 3 else z,
                   v[0].copy(), v[1].copy(), v[2].copy() if dim == 3 else z.copy(), z.copy(), t)


@pytest.mark.parametrize("ktype", [2, 6])
@pytest.mark.parametrize("dim,n,kind", [(2, 1, "clump"), (2, 50, "clump"), (2, 241, "clump"), (3, 17, "clump"),
                                        (3, 250, "clump"), (2, 49152, "lattice"), (2, 49153, "lattice"),
                                        (3, 131072, "lattice"), (3, 131073, "lattice")])
def test_stages_match_the_oracle(hip, oracle, dim, n, kind, ktype):
    case = _cloud(dim, n, kind)
    p = vx.default_params(dim, 1.0)
    p.re_s, p.re_l = (1.9, 1.9) if n > 1000 else (2.1, 3.1)
    p.lambda_ = 0.16832 * p.re_l ** 2
    p.ktype = ktype
    p.turb = 1
    p.dt = 1e-3
    vx.set_box(p, case)
    rng = np.random.default_rng(1)
    fields = {f: rng.normal(0, 1, n) for f in ("U", "V", "W", "P", "PNEW", "PHAT", "UNEW", "VNEW", "WNEW",
                                               "USTAR", "VSTAR", "WSTAR")}
    if dim == 2:
        for f in ("W", "WNEW", "WSTAR"):
            fields[f][:] = 0.0
    sims = [vx.Simulation(p, case, backend=b) for b in (hip, oracle)]
    g, c = sims

    def same(names, what):
        for f in names:
            assert np.array_equal(g.get(f), c.get(f), equal_nan=True), (what, f)

    for s in sims:
        s.init()
        s.set_n0(6.0, 12.0)
        for f, v in fields.items():
            s.set(f, v)
        s.NEIGHBOR()
    for stage, out in (("PNUM", "N"), ("SPS", "NEUT TURB1 TURB2 TURB3"), ("V_FRACTION", "C"),
                       ("PNUMSTAR", "NSTAR"), ("PRESSGRAD", "UNEW VNEW WNEW"), ("COLLISION2", "UNEW VNEW X Y")):
        for s in sims:
            getattr(s, stage)()
        same(out.split(), stage)
        if stage == "PNUM":
            for s in sims:
                for x in "XYZ"[:dim]:
                    s.set(x + "STAR", case.x * 0 + s.get(x))
    q = p.copy()
    q.fluid2_type, q.cohes, q.n_pl, q.meu0 = 1, 1.0, 1.0, 0.85
    for s in sims:
        s.set_params(q)
        for f in ("UNEW", "VNEW", "WNEW"):
            s.set(f, fields[f])
    for s in sims:
        s.VISCOSITY()
    assert np.allclose(g.get("MEU"), c.get("MEU"), rtol=1e-13, atol=0, equal_nan=True)
    for s in sims:
        s.close()
