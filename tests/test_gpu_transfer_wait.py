"""Reading a field back behind enqueued steps: one thread waits for them, not
every thread of the copy."""
import time

import numpy as np
import pytest

from lesamd import api, setup_gen

pytestmark = pytest.mark.gpu


def test_a_download_behind_enqueued_steps_spins_on_one_thread():
    s = setup_gen.build(setup_gen.Workload("wait", 300, 300, 90, dt=0.02, seed=3), dense=False)
    print("\n[transfer wait] 300x300x90", flush=True)
    d = api.Domain(s)
    d.set_graph(True)
    d.run(1, 2, 1000)
    d.download("p")  # the slots exist
    d.run(3, 152, 1000)  # about 0.2 s
    cpu, wall = time.process_time(), time.perf_counter()
    p = d.download("p")
    cpu, wall = time.process_time() - cpu, time.perf_counter() - wall
    # one thread spins for the wait (1 x wall); a second for the runtime's own
    # threads and the copy of 33 MB
    assert cpu < 2.0 * wall, (cpu, wall)
    assert np.isfinite(p).all()
    d.close()
