"""The product that also ends the CG iteration before it (test, beta, new
direction) against the three-kernel form: the same bits, iteration counts and
residuals, when the solve stops at its limit after 1, 2 or 3 iterations, is
read every iteration or in batches, starts warm, refines in mixed precision, has
a zero right-hand side, or takes the learned preconditioner. Product variant 0
is the one form (for the smaller 2D systems the whole solve in one block), 4 the
other; sizes lie around whole blocks of rows and the one block's limits."""
import numpy as np
import pytest

import voxarmps_amd as vx

pytestmark = pytest.mark.gpu


def _solve(s, variant):
    """(error code, pressures, iterations, residual) of the assembled system."""
    s.set_tuning([0, 0, 0, variant])
    code = 0
    try:
        s.CGM()
    except vx.VoxError as e:
        code = e.code
    st = s.status()
    return code, s.get("PNEW"), st.last_iters, st.last_relres


def _same(a, b, what):
    assert a[0] == b[0] and a[2] == b[2], (what, a[0], b[0], a[2], b[2])
    assert np.array_equal(a[1], b[1], equal_nan=True) and a[3] == b[3], what


@pytest.mark.parametrize("shape", [(10, 10, 0), (16, 16, 0), (31, 33, 0), (33, 31, 0), (40, 48, 0), (48, 48, 0), (8, 8, 8), (20, 13, 11)],
                         ids=str)
@pytest.mark.parametrize("precision", [vx._abi.PREC_FP64, vx._abi.PREC_MIXED], ids=["fp64", "mixed"])
def test_fused_and_plain_iterations_agree(hip, shape, precision):
    wx, wy, wz = shape
    dim = 3 if wz else 2
    case = vx.dam_break(dim, 0.005, shape[:dim], (3 * wx, wy + 8, wz + 1)[:dim])
    params = vx.dam3d_params if dim == 3 else vx.dam2d_params
    lattice = vx.Simulation(params(case), case, backend=hip)
    lattice.init()
    n0 = lattice.n0()              # (the jittered maximum leaves hardly any unknown)
    lattice.close()
    case = vx.jitter(case, 0.1 * case.l0, seed=3)
    p = params(case, tol=1e-10)
    p.precision = precision
    s = vx.Simulation(p, case, backend=hip)
    s.init()
    s.set_n0(*n0)
    for st in ("PNUM", "VISCOSITY", "PREDICTION", "PNUMSTAR", "BCON", "MATRIX"):
        getattr(s, st)()
    seen = set()
    for maxit in (1, 2, 3, 400):
        for check in (1, 3):
            for warm in (0, 1):
                q = p.copy()
                q.cg_maxit, q.cg_check, q.warm_start = maxit, check, warm
                s.set_params(q)
                a, b = _solve(s, 4), _solve(s, 0)
                _same(a, b, (maxit, check, warm))
                seen.add(b[0])
    assert 0 in seen and len(seen) == 2            # solved ones and ones at their limit
    s.set_params(p)
    net = vx.LearnedPreconditioner(seed=2, backend=hip)
    net.set_weights(np.random.default_rng(7).uniform(-0.1, 0.1, vx.lpc.NPARAM).astype(np.float32))
    s.attach_lpc(net)
    q = p.copy()
    q.solver = vx._abi.SOLVER_LEARNED_FCG
    s.set_params(q)
    s.CGM()                                        # the Jacobi baseline
    s.MATRIX()
    _same(_solve(s, 4), _solve(s, 0), "learned")
    s.close()
    net.close()


def test_zero_right_hand_side(hip):
    """Pairs one spacing apart whose density is the reference density."""
    n = 600
    x = np.repeat(np.arange(n // 2) * 20.0, 2) + np.tile([0.0, 1.0], n // 2)
    z = np.zeros(n)
    case = vx.Case(2, 1.0, x, z.copy(), z.copy(), z.copy(), z.copy(), z.copy(), z.copy(),
                   np.ones(n, np.int32))
    p = vx.default_params(2, 1.0)
    p.re_s, p.re_l = 2.1, 4.0
    p.lambda_ = 0.16832 * p.re_l ** 2
    p.gx = p.gy = 0.0
    vx.set_box(p, case)
    s = vx.Simulation(p, case, backend=hip)
    s.init()
    for st in ("PNUM", "VISCOSITY", "PREDICTION", "PNUMSTAR"):
        getattr(s, st)()
    s.set_n0(float(s.get("NSTAR")[0]), 1.0)
    s.BCON()
    s.MATRIX()
    assert not s.ppe()["rhs"].any()
    s.MATRIX()
    for v in (4, 0, 0):
        code, pn, it, res = _solve(s, v)
        assert (code, it, res) == (0, 0, 0.0) and not pn.any(), v
    s.close()
