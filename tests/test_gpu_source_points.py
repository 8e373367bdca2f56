"""Source points cost a step nothing on the planes that hold none.

The block that holds the points tests each of its planes for them, and a launch
waits for its slowest block; with one z chunk that block has every plane."""
import time

import numpy as np
import pytest

from cases import hip_prop, make_case

pytestmark = pytest.mark.gpu


def test_time_with_one_and_with_many_points(pyborn):
    import torch

    nx, ny, nz, nt = 192, 192, 600, 150
    cells = nx * ny * nz
    H = hip_prop(pyborn, make_case(32, 32, 32, nt=4, nbound=6))
    H.create_space(10.0, 10.0, 10.0, nx, ny, nz)
    H.set_tuning("source", 2, 2, 4, 1, nz - 8)
    H.set_tuning("rtm_adjoint", 2, 4, 1, 1, nz - 8)
    H.transfer_vel_func1(np.full(cells, 1e-3, np.float32))
    H.transfer_vel_func2(np.full(cells, 1e-3, np.float32))
    at = 70 + nx * (69 + ny * 40)
    H.transfer_receiver_func(1, 1, np.array([at], np.int32), np.zeros((1, nt + 8), np.float32))
    dev = torch.device("cuda:0")
    p0, p1, img = (torch.zeros(cells, device=dev) for _ in range(3))
    tr = torch.zeros((nt + 8, 1), device=dev)
    took = {}
    for points in (1, 32):
        # (one cell in x and y: one block holds them all)
        H.transfer_source_func(np.full(points, at, np.int32),
                               np.ones((points, nt + 8), np.float32))
        for again in (False, True):
            torch.cuda.synchronize()
            t = [time.perf_counter()]
            H.dev_source_prop(1, nt, p0, p1)
            H.synchronize()
            t.append(time.perf_counter())
            H.dev_rtm_adjoint(nt, p1, p0, img, tr)
            H.synchronize()
            t.append(time.perf_counter())
        took[points] = np.diff(t) / nt * 1e6
    H.close()
    print("us per step, source and adjoint:", took)
    assert np.all(took[32] < 1.3 * took[1])
