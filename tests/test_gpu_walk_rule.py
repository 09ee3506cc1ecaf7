"""The list walk that the library picks by itself on both sides of each line of
its rule (particle counts, dimension, cell size): lists are the oracle's."""
import numpy as np
import pytest

import voxarmps_amd as vx

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dim,n,ks,kl", [(2, 65536, 2.1, 3.1), (2, 65537, 2.1, 3.1), (3, 49152, 2.1, 3.1),
                                         (3, 49153, 2.1, 3.1), (3, 98304, 3.0, 3.0), (3, 98305, 3.0, 3.0),
                                         (3, 262144, 1.6, 1.6), (3, 262145, 1.6, 1.6)])
def test_lists_on_both_sides_of_the_rule(hip, oracle, dim, n, ks, kl):
    rng = np.random.default_rng(n)
    side = int(np.ceil(n ** (1 / dim)))
    k = np.arange(n)
    pos = [k % side, k // side % side, k // side ** 2][:dim]
    pos = [p + rng.uniform(-0.1, 0.1, n) for p in pos]
    z = np.zeros(n)
    case = vx.Case(dim, 1.0, pos[0], pos[1], pos[2] if dim == 3 else z, z.copy(), z.copy(), z.copy(), z.copy(),
                   np.ones(n, np.int32))
    p = vx.default_params(dim, 1.0)
    p.re_s, p.re_l = ks, kl
    p.lambda_ = 0.16832 * p.re_l ** 2
    vx.set_box(p, case)
    g, c = (vx.Simulation(p, case, backend=b) for b in (hip, oracle))
    g.NEIGHBOR()
    c.NEIGHBOR()
    for w in (vx.LIST_S, vx.LIST_L):
        assert np.array_equal(g.cells(w), c.cells(w))
        for a, b in zip(g.neighbors(w), c.neighbors(w)):
            assert np.array_equal(a, b)
    g.close()
    c.close()
