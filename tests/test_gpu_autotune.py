"""The autotuner on a context whose last search ended with a particle outside the box:
its own searches report what they find, not what the earlier one did."""
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
