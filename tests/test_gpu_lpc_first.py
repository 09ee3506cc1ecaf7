"""The first pass on fresh memory gives what later ones give: the learned solve after
the Jacobi baseline, and the gradient on a system dumped into a new network, on
systems whose buffers take longer to clear than the first kernels take to start."""
import os

import numpy as np
import pytest

import voxarmps_amd as vx

pytestmark = pytest.mark.gpu

WEIGHTS = os.path.join(os.path.dirname(vx.__file__), "data", "lpc_weights.npy")


def _sim(hip, shape):
    case = vx.dam_break(3, 0.005, shape, (16 * shape[0] // 5, shape[1] + 12, shape[2] + 1))
    p = vx.dam3d_params(case, tol=1e-8)
    s = vx.Simulation(p, case, backend=hip)
    s.init()
    for st in ("PNUM", "VISCOSITY", "PREDICTION", "PNUMSTAR", "BCON"):
        getattr(s, st)()
    return s, p


@pytest.mark.parametrize("shape", [(24, 24, 20), (50, 60, 56)], ids=str)
def test_first_learned_solve(hip, shape):
    seen = []
    for _ in range(3):
        s, p = _sim(hip, shape)
        net = vx.LearnedPreconditioner(backend=hip)
        net.set_weights(np.load(WEIGHTS, allow_pickle=False))
        s.attach_lpc(net)
        q = p.copy()
        q.solver = vx._abi.SOLVER_LEARNED_FCG
        s.set_params(q)
        s.PRESSURECALC()                           # the Jacobi baseline
        for _ in range(2):
            info = s.PRESSURECALC()
            seen.append((info.iterations, info.relres, s.get("PNEW")))
        assert s.status().lpc_fallbacks == 0
        s.close()
        net.close()
    for it, res, pn in seen[1:]:
        assert (it, res) == seen[0][:2] and np.array_equal(pn, seen[0][2])


def test_first_gradient(hip):
    s, _ = _sim(hip, (44, 48, 44))
    s.MATRIX()
    seen = []
    for _ in range(2):
        net = vx.LearnedPreconditioner(backend=hip)
        net.set_weights(np.load(WEIGHTS, allow_pickle=False))
        for i in range(2):
            index = net.dump(s)
            assert index == i
        for index in (0, 1, 0):
            seen.append(net.loss_grad(index, 12345))
        net.close()
    for loss, grad in seen[1:]:
        assert loss == seen[0][0] and np.array_equal(grad, seen[0][1])
    s.close()
