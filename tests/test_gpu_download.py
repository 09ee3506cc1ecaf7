"""Downloads through the pinned buffer: sizes around its pieces (256 kB), the
helpers' threshold (1 MB) and the buffer itself (16 MB), 4- and 8-byte fields,
pageable and pinned destinations, and several threads on one context."""
import ctypes as C
import threading

import numpy as np
import pytest
import torch

import voxarmps_amd as vx
from voxarmps_amd.sim import F

pytestmark = pytest.mark.gpu


def _sim(hip, n):
    side = int(np.ceil(np.sqrt(n)))
    k = np.arange(n)
    z = np.zeros(n)
    rng = np.random.default_rng(n)
    case = vx.Case(2, 1.0, (k % side).astype(float), (k // side).astype(float), z,
                   rng.normal(size=n), rng.normal(size=n), z.copy(), rng.normal(size=n),
                   rng.integers(0, 3, n).astype(np.int32))
    p = vx.default_params(2, 1.0)
    vx.set_box(p, case)
    return vx.Simulation(p, case, backend=hip), case


@pytest.mark.parametrize("n", [1, 2, 3, 511, 32767, 32768, 32769, 65537, 131071, 131073, 1200001,
                               2097152, 2097155])
def test_download_returns_what_was_uploaded(hip, n):
    s, case = _sim(hip, n)
    for _ in range(2):
        for name, want in (("U", case.u), ("PTYPE", case.ptype), ("P", case.p), ("V", case.v)):
            assert np.array_equal(s.get(name), want), name
    pinned = torch.empty(n, dtype=torch.float64, pin_memory=True)
    hip.check(hip.fn("download")(s.ctx, F["U"], C.c_void_p(pinned.data_ptr())), "download")
    assert np.array_equal(pinned.numpy(), case.u)
    s.close()


def test_threads_share_a_context(hip):
    s, case = _sim(hip, 300000)
    wrong = []

    def reader(name, want):
        for _ in range(20):
            if not np.array_equal(s.get(name), want):
                wrong.append(name)

    ts = [threading.Thread(target=reader, args=a) for a in
          (("U", case.u), ("V", case.v), ("P", case.p), ("PTYPE", case.ptype))]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    assert not wrong
    s.close()
