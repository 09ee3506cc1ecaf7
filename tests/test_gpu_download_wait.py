"""A download behind long queued work: its helper threads sleep until the data are on
their way, and only the caller waits in the runtime (less than 1.5 times the wall
time in CPU time; helpers that spin make it 3), and the values are those of the
queued work."""
import time

import numpy as np
import pytest

import voxarmps_amd as vx

pytestmark = pytest.mark.gpu


def test_waiting_download_leaves_the_cores(hip):
    case = vx.dam_break(3, 0.005, (44, 44, 36), (140, 53, 37))
    s = vx.Simulation(vx.dam3d_params(case), case, backend=hip)
    assert 8 * s.tp >= 1 << 20
    s.init()
    for st in ("PNUM", "VISCOSITY", "PREDICTION"):
        getattr(s, st)()
    want = s.get("USTAR")
    for _ in range(1500):
        s.PREDICTION()
    cpu, wall = time.process_time(), time.perf_counter()
    got = s.get("USTAR")
    cpu, wall = time.process_time() - cpu, time.perf_counter() - wall
    print(f"waited {wall * 1e3:.0f} ms, {cpu * 1e3:.0f} ms of CPU time")
    assert wall > 0.05 and cpu < 1.5 * wall
    assert np.array_equal(got, want)
    s.close()
