"""What a call with large host results costs the host while the GPU works.

The calls queue the whole time loop and then wait for the result's first
bytes; only from then on have the copying threads anything to do."""
import time

import numpy as np
import pytest

from cases import hip_prop, make_case

pytestmark = pytest.mark.gpu


def test_no_thread_polls_for_the_time_loop(pyborn):
    # 131 MB results after 2000 steps of about 100 us, all of them queued
    n, nt = 320, 2000
    c = make_case(48, 48, 48, nt=40, nbound=6)
    H = hip_prop(pyborn, c)
    H.create_space(*c.d, n, n, n)
    H.transfer_source_func(np.array([n // 2 + n * (n // 2 + n * 40)], np.int32),
                           np.ones((1, nt + 8), np.float32))
    H.transfer_vel_func1(np.full(n**3, 1e-3, np.float32))
    p0, p1 = np.zeros(n**3, np.float32), np.zeros(n**3, np.float32)
    H.source_prop(p0, p1, 1, 8)  # launch shapes, buffers, the pinned ring
    assert np.abs(p0).max() > 0
    p0[:], p1[:] = 0, 0
    wall, cpu = time.perf_counter(), time.process_time()
    H.source_prop(p0, p1, 1, nt)
    wall, cpu = time.perf_counter() - wall, time.process_time() - cpu
    H.close()
    print("wall %.3f s, processor %.3f s" % (wall, cpu))
    assert wall > 0.1
    # the calling thread and one of the runtime's; four polling ones make it 5
    assert cpu < 2.5 * wall
