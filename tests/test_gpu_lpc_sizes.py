"""The network on systems past the sizes where its kernels change form - weight
gradients in chunks of more than 64 rows (above 16,384 rows, here no multiple of 4)
and the aggregation with 4 lanes a row (from 32,768 rows) - against the FP64 oracle.

Tolerances: the oracle makes the same bf16 roundings of FP64 sums, this library of
FP32 sums. A sum of 64 terms is off by some 5e-7 of its size, so about 3e-4 of the
activations round to the other neighbour, 2^-8 away: 7e-5 of a layer in L2, some
3e-4 after four layers. The gradient's FP32 sums add less. 5e-3 in L2 for each block of
parameters leaves a factor ten; single outputs keep the 3e-2 (1e-3 in the median)
of the small systems."""
import numpy as np
import pytest

import voxarmps_amd as vx
from oracle import lpc as olpc
from test_gpu_cg_sizes import lattice_system
from test_gpu_lpc import oracle_system, random_weights

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [16387, 32767, 32771])
def test_network_matches_the_oracle(hip, n):
    s, case, p = lattice_system(hip, 2, n, 2.1, rl=3.1)
    S, _ = oracle_system(s, case, p)
    assert S.nu == n
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
    k = 0
    for name, shape in olpc.LAYOUT:
        e = k + int(np.prod(shape))
        err = np.linalg.norm(grad[k:e] - go[k:e]) / np.linalg.norm(go[k:e])
        print(f"{name}: {err:.1e}")
        assert err <= 5e-3, name
        k = e
    s.close()
    net.close()
