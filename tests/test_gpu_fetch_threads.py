"""Threads that share a context and read its status at the same time: every call
returns, with the counts of the state."""
import threading

import numpy as np
import pytest

import voxarmps_amd as vx

pytestmark = pytest.mark.gpu


def test_threads_read_the_status_of_one_context(hip):
    case = vx.dam_break(2, 0.01, (25, 50), (100, 70))
    s = vx.Simulation(vx.dam2d_params(case), case, backend=hip)
    s.init()
    s.step(3)
    before = [s.get(f) for f in "XYUVP"]
    errors = []

    def work():
        try:
            for _ in range(3000):
                s.PREPDATA()
        except vx.VoxError as e:
            errors.append(str(e))

    threads = [threading.Thread(target=work) for _ in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not errors
    s.PREPDATA()
    st = s.status()
    assert st.nan_count == 0 and st.out_of_box == 0
    for f, a in zip("XYUVP", before):
        assert np.array_equal(s.get(f), a)
    s.close()
