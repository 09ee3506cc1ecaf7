"""Searches that end without room for their rows: a clump whose rows no device could
store, and rows longer than the storage in a search that ends on a particle outside the
box. The stages that follow find empty rows, and the next search of good positions
gives the oracle's lists at once."""
import numpy as np
import pytest

import voxarmps_amd as vx

pytestmark = pytest.mark.gpu


def _lattice(n):
    side = int(np.ceil(np.sqrt(n)))
    k = np.arange(n)
    rng = np.random.default_rng(n)
    z = np.zeros(n)
    return vx.Case(2, 1.0, k % side + rng.uniform(-0.2, 0.2, n), k // side + rng.uniform(-0.2, 0.2, n), z,
                   z.copy(), z.copy(), z.copy(), z.copy(), np.ones(n, np.int32))


def _pair(hip, oracle, case, ks, kl, mode):
    p = vx.default_params(2, 1.0)
    p.re_s, p.re_l = ks, kl
    p.lambda_ = 0.16832 * p.re_l ** 2
    p.list_mode = mode
    vx.set_box(p, case)
    sims = [vx.Simulation(p, case, backend=b) for b in (hip, oracle)]
    for s in sims:
        s.init()
    return sims


def _same_lists(g, c, case, two):
    for s in (g, c):
        s.set("X", case.x + 0.05)
        s.set("Y", case.y)
        s.NEIGHBOR()
        s.PNUM()
    assert np.array_equal(g.get("N"), c.get("N"))
    for w in (vx.LIST_S, vx.LIST_L)[:1 + two]:
        for a, b in zip(g.neighbors(w), c.neighbors(w)):
            assert np.array_equal(a, b)


def test_clump_beyond_any_memory(hip, oracle):
    """270,000 particles within one radius: rows of 364 GB on a card of 288 GB."""
    n = 270000
    case = _lattice(n)
    g, c = _pair(hip, oracle, case, 2.1, 2.1, 1)
    for repeat in range(2):
        g.set("X", 100.0 + 0.5 * np.sin(np.arange(n)))
        g.set("Y", 100.0 + 0.5 * np.cos(np.arange(n)))
        with pytest.raises(vx.VoxError) as e:
            g.NEIGHBOR()
        assert e.value.code == vx._abi.VOX_ERR_HIP and "neighbour rows" in str(e.value)
        g.PNUM()
        assert not g.get("N").any()
        assert not g.neighbors(vx.LIST_S)[0].any()
    _same_lists(g, c, case, False)
    for s in (g, c):
        s.close()


@pytest.mark.parametrize("mode", [0, 1, 2])
@pytest.mark.parametrize("ks,kl", [(2.1, 2.1), (2.1, 3.1)], ids=str)
def test_long_rows_and_a_particle_outside(hip, oracle, mode, ks, kl):
    n = 3000
    case = _lattice(n)
    g, c = _pair(hip, oracle, case, ks, kl, mode)
    x, y = case.x.copy(), case.y.copy()
    x[:2000] = 20.0 + 0.5 * np.sin(np.arange(2000))
    y[:2000] = 20.0 + 0.5 * np.cos(np.arange(2000))
    x[-1] = 1e6
    g.set("X", x)
    g.set("Y", y)
    with pytest.raises(vx.VoxError) as e:
        g.NEIGHBOR()
    assert e.value.code == vx._abi.VOX_ERR_DOMAIN
    for st in ("PNUM", "V_FRACTION", "VISCOSITY", "PREDICTION", "PNUMSTAR"):
        getattr(g, st)()
    assert not g.get("N").any()
    _same_lists(g, c, case, kl != ks)
    for s in (g, c):
        s.close()
