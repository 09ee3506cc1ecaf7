"""The autotuner on a context whose last search ended with a particle outside the box:
its own searches report what they find, not what the earlier one did. And on systems
whose solve does more in product 0 than a product (one block, or the direction
renewed in it): that product stays, whatever was set before."""
import numpy as np
import pytest

import voxarmps_amd as vx

pytestmark = pytest.mark.gpu


def test_autotune_after_a_domain_error(hip, oracle):
    case = vx.dam_break(2, 0.01, (20, 24), (60, 40))
    p = vx.dam2d_params(case)
    g, c = (vx.Simulation(p, case, backend=b) for b in (hip, oracle))
    for s in (g, c):
        s.init()
    x = case.x.copy()
    x[-1] = 1e3
    g.set("X", x)
    with pytest.raises(vx.VoxError) as e:
        g.NEIGHBOR()
    assert e.value.code == vx._abi.VOX_ERR_DOMAIN
    with pytest.raises(vx.VoxError) as e:
        g.autotune(reps=1)
    assert e.value.code == vx._abi.VOX_ERR_DOMAIN
    g.set("X", case.x)
    g.autotune(reps=2)
    c.NEIGHBOR()
    g.NEIGHBOR()
    for w in (vx.LIST_S, vx.LIST_L):
        for a, b in zip(g.neighbors(w), c.neighbors(w)):
            assert np.array_equal(a, b)
    for s in (g, c):
        s.close()


@pytest.mark.parametrize("dim,shape,tank", [(2, (25, 50), (100, 70)), (2, (400, 300), (1600, 320)),
                                            (3, (20, 20, 16), (64, 24, 17))], ids=str)
@pytest.mark.parametrize("precision", [vx._abi.PREC_FP64, vx._abi.PREC_MIXED], ids=["fp64", "mixed"])
def test_fused_solves_keep_their_product(hip, dim, shape, tank, precision):
    case = vx.dam_break(dim, 0.01 if dim == 2 else 0.005, shape, tank)
    p = (vx.dam3d_params if dim == 3 else vx.dam2d_params)(case)
    p.precision = precision
    a, b = (vx.Simulation(p, case, backend=hip) for _ in range(2))
    for s in (a, b):
        s.init()
    b.set_tuning([0, 0, 8, 4])
    b.autotune(reps=5)
    assert b.tuning()[3] == 0
    for s in (a, b):
        s.step(2)
    for f in "XYUVP":
        assert np.array_equal(a.get(f), b.get(f)), f
    for s in (a, b):
        s.close()
