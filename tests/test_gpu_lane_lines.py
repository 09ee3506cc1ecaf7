"""Both sides of the lines between one thread and 16 lanes per particle that depend on
the length of a row: lists against the oracle, and the stages against the oracle bit
for bit (the Herschel-Bulkley viscosity, whose line is three quarters of the other
stages', to 1e-13: pow)."""
import numpy as np
import pytest

import voxarmps_amd as vx
from test_gpu_stage_lanes import _cloud, test_stages_match_the_oracle as stages_match
from test_gpu_walk_rule import test_lists_on_both_sides_of_the_rule as lists_match

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dim,n,ks,kl", [(2, 98304, 2.6, 3.1), (2, 98305, 2.6, 3.1), (3, 98304, 1.6, 2.1),
                                         (3, 98305, 1.6, 2.1), (3, 262144, 2.5, 2.5), (3, 262145, 2.5, 2.5)])
def test_lists(hip, oracle, dim, n, ks, kl):
    lists_match(hip, oracle, dim, n, ks, kl)


@pytest.mark.parametrize("dim,n", [(2, 36864), (2, 36865), (3, 73728), (3, 73729), (3, 98304), (3, 98305)])
def test_stages(hip, oracle, dim, n):
    """rows of 11 (2D) and 29 (3D) entries"""
    stages_match(hip, oracle, dim, n, "lattice", 2)


@pytest.mark.parametrize("n", [98304, 98305, 131072, 131073])
def test_stages_of_long_rows(hip, oracle, n):
    """2D rows of 50 entries"""
    case = _cloud(2, n, "lattice")
    p = vx.default_params(2, 1.0)
    p.re_s = p.re_l = 4.0
    p.lambda_ = 0.16832 * p.re_l ** 2
    p.turb, p.dt = 1, 1e-3
    p.fluid2_type, p.cohes, p.n_pl, p.meu0 = 1, 1.0, 1.0, 0.85
    vx.set_box(p, case)
    sims = [vx.Simulation(p, case, backend=b) for b in (hip, oracle)]
    g, c = sims
    rng = np.random.default_rng(2)
    fields = {f: rng.normal(0, 1, n) for f in ("UNEW", "VNEW", "PNEW", "PHAT")}
    for s in sims:
        s.init()
        for f, v in fields.items():
            s.set(f, v)
    for stage, out in (("PNUM", "N"), ("SPS", "NEUT TURB1 TURB2"), ("V_FRACTION", "C"), ("VISCOSITY", "MEU"),
                       ("PRESSGRAD", "UNEW VNEW"), ("COLLISION2", "UNEW VNEW X Y")):
        for s in sims:
            getattr(s, stage)()
        for f in out.split():
            if f == "MEU":
                assert np.allclose(g.get(f), c.get(f), rtol=1e-13, atol=0, equal_nan=True)
            else:
                assert np.array_equal(g.get(f), c.get(f), equal_nan=True), (stage, f)
    for s in sims:
        s.close()
