"""The network's row walks, matrix-core gradients and strong couplings at sizes
around their tiles (16 rows a tile, 64 rows a block, 8 entries a batch, weight
gradients over chunks of 64 rows) and with more strong couplings per row than
wait on chip, against the FP64 oracle with the tolerances of the 2D test system
(bf16 operands bound them)."""
import numpy as np
import pytest

import voxarmps_amd as vx
from oracle import lpc as olpc
from test_gpu_lpc import oracle_system, random_weights

pytestmark = pytest.mark.gpu


def _system(hip, shape, dl):
    wx, wy, wz = shape
    dim = 3 if wz else 2
    case = vx.dam_break(dim, 0.005, shape[:dim], (2 * wx + 3, wy + 6, wz + 1)[:dim])
    lattice = vx.Simulation((vx.dam3d_params if dim == 3 else vx.dam2d_params)(case), case, backend=hip)
    lattice.init()
    n0 = lattice.n0()
    lattice.close()
    case = vx.jitter(case, 0.1 * case.l0, seed=5)
    p = (vx.dam3d_params if dim == 3 else vx.dam2d_params)(case, tol=1e-9)
    p.dl = dl * case.l0
    s = vx.Simulation(p, case, backend=hip)
    s.init()
    s.set_n0(*n0)
    for st in ("PNUM", "NEIGHBOR", "VISCOSITY", "PREDICTION", "PNUMSTAR", "BCON", "MATRIX"):
        getattr(s, st)()
    return s, case, p


@pytest.mark.parametrize("shape,dl", [((6, 6, 0), 1.0), ((15, 17, 0), 1.0), ((33, 31, 0), 1.6),
                                      ((9, 8, 8), 1.0), ((13, 12, 11), 1.5)], ids=str)
def test_rows_and_gradients_match_the_oracle(hip, shape, dl):
    s, case, p = _system(hip, shape, dl)
    S, P = oracle_system(s, case, p)
    net = vx.LearnedPreconditioner(seed=1, backend=hip)
    idx = net.dump(s)
    w = random_weights(5)
    net.set_weights(w)
    f, g, c = net.eval(idx, S.nu)
    assert np.max(np.abs(f - S.f)) <= 1e-5 * max(1.0, np.max(np.abs(S.f)))
    st = olpc.forward(w.astype(np.float64), S)
    for got, want in ((g, st["g"]), (c, st["c"])):
        rel = np.abs(got - want) / np.abs(want)
        assert np.median(rel) <= 1e-3 and rel.max() <= 3e-2
    L, grad = net.loss_grad(idx, 12345)
    Lo, go = olpc.loss_grad(w.astype(np.float64), S, S.probes(12345), rounding=True)
    assert L == pytest.approx(Lo, rel=1e-3)
    assert np.linalg.norm(grad - go) <= 3e-2 * np.linalg.norm(go)
    L2, again = net.loss_grad(idx, 12345)
    assert L2 == L and np.array_equal(again, grad)
    # the context's own couplings: the learned solve meets the tolerance and
    # agrees with Jacobi-CG
    s.MATRIX()
    s.CGM()
    pj = s.get("PNEW")
    net.set_weights(random_weights(7, scale=0.05))
    s.attach_lpc(net)
    p.solver = vx._abi.SOLVER_LEARNED_FCG
    s.set_params(p)
    s.CGM()
    info = s.CGM()
    assert info.converged and info.relres <= 1e-9
    assert np.linalg.norm(s.get("PNEW") - pj) <= 1e-6 * np.linalg.norm(pj)
    s.close()
    net.close()
