"""The stages that read a row 16 entries at a time (predictor, PPE assembly) at
the sizes where that can go wrong: row lengths around multiples of 16, rows that
end while others of the wave go on, rows longer than the predictor's queue,
empty rows, few particles, rows whose columns are mostly dropped, and pairs at
exactly the radius and one unit in the last place inside it. The same
operations in the same order as the oracle's: equal bits."""
import numpy as np
import pytest

import voxarmps_amd as vx

pytestmark = pytest.mark.gpu

OUT = ("XSTAR", "YSTAR", "ZSTAR", "USTAR", "VSTAR", "WSTAR")


def _cloud(pos, dim, rng):
    n = len(pos)
    z = np.zeros(n)
    v = rng.normal(0, 1, (3, n))
    return vx.Case(dim, 1.0, pos[:, 0].copy(), pos[:, 1].copy(),
                   pos[:, 2].copy() if dim == 3 else z, v[0].copy(), v[1].copy(),
                   v[2].copy() if dim == 3 else z.copy(), z.copy(),
                   rng.choice(np.array([-1, 0, 1, 1, 1, 2], np.int32), n))


def _lattice(dim, shape):
    return np.stack(np.meshgrid(*[np.arange(float(s)) for s in shape], indexing="ij"),
                    -1).reshape(-1, dim)


def _cases():
    for dim in (2, 3):
        rng = np.random.default_rng(dim)
        for n in (1, 5, 33, 400, 1201):
            side = n ** (1 / dim) * 0.8
            yield f"{dim}d-random-{n}", _cloud(rng.uniform(0, side, (n, dim)), dim, rng)
        grid = _lattice(dim, (9, 11, 13)[:dim])
        yield f"{dim}d-at-radius", _cloud(grid, dim, rng)
        yield f"{dim}d-inside-radius", _cloud(grid * (1 - 2.0 ** -53), dim, rng)
        clump = np.concatenate([rng.uniform(0, 0.9, (90, dim)) + 3.0, rng.uniform(0, 8, (150, dim)),
                                rng.uniform(0, 60, (40, dim))])
        yield f"{dim}d-clump", _cloud(clump, dim, rng)


@pytest.mark.parametrize("name,case", list(_cases()), ids=lambda v: v if isinstance(v, str) else "")
@pytest.mark.parametrize("ktype", [1, 2, 6])
def test_rows_match_the_oracle(hip, oracle, name, case, ktype):
    dim, n = case.dim, case.tp
    p = vx.default_params(dim, 1.0)
    p.re_s, p.re_l = 2.0, 3.0
    p.lambda_ = 0.16832 * p.re_l ** 2
    p.ktype = ktype
    vx.set_box(p, case)
    rng = np.random.default_rng(n)
    fields = {f: rng.normal(0, 1, n) for f in ("U", "V", "W", "PHAT", "PNEW", "UNEW", "VNEW", "WNEW")}
    if dim == 2:
        fields["W"][:] = fields["WNEW"][:] = 0.0
    sims = [vx.Simulation(p, case, backend=b) for b in (hip, oracle)]
    g, c = sims
    for s in sims:
        s.init()
        s.set_n0(5.0, 9.0)
        for f, v in fields.items():
            s.set(f, v)
        s.NEIGHBOR()
        s.PNUM()
        s.VISCOSITY()
    eddy = rng.uniform(0, 1e-3, n) * (rng.random(n) < 0.5)
    meu = rng.uniform(0.5e-3, 2e-3, n)
    for what, sets in (("one viscosity", {}), ("eddy", {"NEUT": eddy}), ("general", {"MEU": meu})):
        for s in sims:
            for f, v in sets.items():
                s.set(f, v)
        c.PREDICTION()
        for v in (8, 6, 0):
            g.set_tuning([0, 0, v, 0])
            g.PREDICTION()
            for f in OUT:
                assert np.array_equal(g.get(f), c.get(f)), (what, v, f)
    for s in sims:
        s.PNUMSTAR()
    bcon = rng.integers(0, 3, n).astype(np.int32)
    for keep in ("BCON", "few"):
        for s in sims:
            s.BCON()
            if keep == "few":                      # most columns are dropped
                s.set("BCON", np.where(c.get("BCON") == 0, np.minimum(bcon, 1), c.get("BCON")))
        for matopt in (0, 1):
            q = p.copy()
            q.matopt = matopt
            a = []
            for s in sims:
                s.set_params(q)
                s.MATRIX()
                a.append(s.ppe())
            for k in ("rowptr", "cols", "vals", "rhs", "ids"):
                assert np.array_equal(a[0][k], a[1][k]), (keep, matopt, k)
    for s in sims:
        s.close()
