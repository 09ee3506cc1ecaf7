"""The forms of a CG iteration against each other at the sizes where the number of
product blocks changes how their partial sums are added: 64 blocks (one register a
lane), 512 (each wave adds for itself), 768 (up to which any product renews the
direction), above that a 2D system (few columns a window: renewed too) and a 3D one
(not), the last two past the bytes that stay in cache. Product variant 0 is the one
form, 4 the other; pressures, iterations and residuals are the same bits, stopped
at a limit and at the tolerance, in FP64, mixed precision and with the learned
preconditioner."""
import numpy as np
import pytest

import voxarmps_amd as vx

pytestmark = pytest.mark.gpu


def lattice_system(backend, dim, n, re, precision=vx._abi.PREC_FP64, rl=None):
    """n jittered fluid particles, all of them unknowns (the density asked of a
    particle below the surface is 1, a lattice corner has more), at a time step
    whose diagonal shift makes the system well conditioned; MATRIX has run."""
    rng = np.random.default_rng(n)
    side = int(np.ceil(n ** (1 / dim)))
    k = np.arange(n)
    pos = [q + rng.uniform(-0.1, 0.1, n) for q in (k % side, k // side % side, k // side ** 2)[:dim]]
    z = np.zeros(n)
    case = vx.Case(dim, 1.0, pos[0], pos[1], pos[2] if dim == 3 else z, z.copy(), z.copy(), z.copy(), z.copy(),
                   np.ones(n, np.int32))
    p = vx.default_params(dim, 1.0)
    p.re_s = p.re_l = re
    if rl:
        p.re_l = rl
    p.lambda_ = 0.16832 * p.re_l ** 2
    p.dt = 4e-3
    p.cg_tol = 1e-9
    p.precision = precision
    vx.set_box(p, case)
    s = vx.Simulation(p, case, backend=backend)
    s.init()
    n0l = s.n0()[1]
    s.set_n0(1.0, n0l)
    for st in ("PNUM", "VISCOSITY", "PREDICTION", "PNUMSTAR", "BCON", "MATRIX"):
        getattr(s, st)()
    return s, case, p


def _solve(s, variant):
    s.set_tuning([0, 0, 8, variant])
    code = 0
    try:
        s.CGM()
    except vx.VoxError as e:
        code = e.code
    st = s.status()
    return code, s.get("PNEW"), st.last_iters, st.last_relres


def _compare(s, what):
    a, b = _solve(s, 4), _solve(s, 0)
    assert a[0] == b[0] and a[2] == b[2] and a[3] == b[3], (what, a[0], b[0], a[2:], b[2:])
    assert np.array_equal(a[1], b[1], equal_nan=True), what
    return b


SIZES = [(2, 16384, 2.1), (2, 16385, 2.1), (2, 131072, 2.1), (2, 131073, 2.1), (2, 196608, 2.1), (2, 196609, 2.1),
         (2, 600000, 4.1), (3, 262144, 3.7)]


@pytest.mark.parametrize("dim,n,re", SIZES, ids=str)
@pytest.mark.parametrize("precision", [vx._abi.PREC_FP64, vx._abi.PREC_MIXED], ids=["fp64", "mixed"])
def test_product_forms_agree(hip, dim, n, re, precision):
    s, _, p = lattice_system(hip, dim, n, re, precision)
    seen = set()
    for maxit in (1, 2, 400):
        q = p.copy()
        q.cg_maxit = maxit
        s.set_params(q)
        code, pn, iters, _ = _compare(s, (dim, n, maxit))
        seen.add(code)
        assert pn.any()
    assert seen == {0, vx._abi.VOX_ERR_SOLVER} and iters > 3
    assert np.count_nonzero(s.get("BCON")) == 0
    s.close()


@pytest.mark.parametrize("n", [131072, 131073, 196608, 196609])
def test_learned_forms_agree(hip, n):
    s, _, p = lattice_system(hip, 2, n, 2.1)
    net = vx.LearnedPreconditioner(seed=2, backend=hip)
    net.set_weights(np.random.default_rng(7).uniform(-0.1, 0.1, vx.lpc.NPARAM).astype(np.float32))
    s.attach_lpc(net)
    q = p.copy()
    q.solver = vx._abi.SOLVER_LEARNED_FCG
    s.set_params(q)
    s.CGM()                                        # the Jacobi baseline
    s.MATRIX()
    code, pn, iters, _ = _compare(s, n)
    assert code == 0 and iters > 2 and pn.any() and s.status().lpc_fallbacks == 0
    s.close()
    net.close()
