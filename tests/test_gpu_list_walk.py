"""The matrix-core list walk at the sizes where it can go wrong: fewer particles
than a wave, a wave that straddles rows of cells, runs of candidates around the
16- and 64-candidate blocks, many pairs exactly at the radius (which FP32 cannot
decide), clumps whose rows outgrow their capacity, and very small and large
coordinates. Lists and cells are the oracle's, entry for entry."""
import numpy as np
import pytest

import voxarmps_amd as vx

pytestmark = pytest.mark.gpu


def _cloud(pos, dim, l0):
    n = len(pos)
    z = np.zeros(n)
    return vx.Case(dim, l0, pos[:, 0].copy(), pos[:, 1].copy(),
                   pos[:, 2].copy() if dim == 3 else z.copy(), z.copy(), z.copy(), z.copy(),
                   z.copy(), np.ones(n, np.int32))


def _lattice(dim, shape, l0):
    g = np.stack(np.meshgrid(*[np.arange(s) for s in shape], indexing="ij"), -1).reshape(-1, dim)
    return g * l0


def _cases():
    rng = np.random.default_rng(5)
    for dim in (2, 3):
        for n in (1, 15, 17, 63, 65, 129, 1000):
            yield f"{dim}d-random-{n}", _cloud(rng.uniform(0, 6, (n, dim)), dim, 1.0), 2.1, 4.0
        # pairs at exactly 2 and 4 spacings: several hundred per wave
        yield f"{dim}d-at-radius", _cloud(_lattice(dim, (9, 13, 21)[:dim], 1.0), dim, 1.0), 2.0, 4.0
        # 300 particles in a ball of half a spacing: rows past any capacity
        clump = np.concatenate([rng.uniform(0, 0.5, (300, dim)) + 3.0, rng.uniform(0, 8, (200, dim))])
        yield f"{dim}d-clump", _cloud(clump, dim, 1.0), 2.1, 4.0
        # one long row of cells along each axis
        for a in range(dim):
            line = rng.uniform(0, 0.5, (700, dim))
            line[:, a] *= 150.0
            yield f"{dim}d-line-{a}", _cloud(line, dim, 1.0), 2.1, 3.2
        for scale, shift in ((1e-9, 0.0), (1e7, -3e8), (1.0, 1e4)):
            yield (f"{dim}d-scale-{scale:g}-{shift:g}",
                   _cloud(rng.uniform(0, 7, (500, dim)) * scale + shift, dim, scale), 2.1, 4.0)


@pytest.mark.parametrize("name,case,ks,kl", list(_cases()), ids=lambda v: v if isinstance(v, str) else "")
@pytest.mark.parametrize("delta", [0.2, 1.5], ids=["delta", "wide-delta"])
def test_walks_match_the_oracle(hip, oracle, name, case, ks, kl, delta):
    p = vx.default_params(case.dim, case.l0)
    p.re_s, p.re_l = ks * case.l0, kl * case.l0
    p.lambda_ = 0.16832 * p.re_l ** 2
    p.delta = delta * case.l0
    vx.set_box(p, case)
    c = vx.Simulation(p, case, backend=oracle)
    c.NEIGHBOR()
    want = {w: (c.cells(w), *c.neighbors(w)) for w in (vx.LIST_S, vx.LIST_L)}
    for mode in (1, 2):
        p.list_mode = mode
        g = vx.Simulation(p, case, backend=hip)
        g.NEIGHBOR()
        for w, (cells, cnt, ids) in want.items():
            assert np.array_equal(g.cells(w), cells), (mode, w)
            got = g.neighbors(w)
            assert np.array_equal(got[0], cnt), (mode, w)
            assert np.array_equal(got[1], ids), (mode, w)
        # list L's own rows (before the export above replaces compact ones)
        g.NEIGHBOR()
        c.NEIGHBOR()
        g.init()
        c.init()
        assert g.n0() == c.n0()
        g.close()
    c.close()
