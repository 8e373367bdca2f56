"""A batch whose forward found no memory for its levels.

The level buffers of a batch grow when 24-bit levels of s and r, 6 bytes per
cell, take the place of FP32 ones.  A forward that cannot have them fails with
BORN_ERR_NOMEM; the batch is then as good as before for what does fit."""
import numpy as np
import pytest

from cases import hip_prop, make_case

pytestmark = pytest.mark.gpu


def _fill(torch, leave):
    """device memory down to `leave` bytes, as a list of tensors"""
    held, size = [], 8 << 30
    while size >= 16 << 20:
        free = torch.cuda.mem_get_info()[0]
        if free - size < leave:
            size //= 2
            continue
        held.append(torch.empty(size, dtype=torch.uint8, device="cuda:0"))
    return held


def test_adjoint_after_a_forward_without_memory(pyborn):
    import torch

    nx, ny, nz, nt = 304, 304, 288, 6
    cells = nx * ny * nz
    rng = np.random.default_rng(4)
    at = 150 + nx * (140 + ny * 50)
    shot = {"nx": nx, "ny": ny, "nz": nz, "vel": np.full(cells, 4.0, np.float32),
            "model": rng.standard_normal(cells).astype(np.float32),
            "src_locs": np.array([at], np.int32),
            "src_vals": np.ones((1, nt + 8), np.float32), "rec_nx": 4, "rec_ny": 1,
            "rec_locs": np.arange(at, at + 4, dtype=np.int32)}
    H = hip_prop(pyborn, make_case(32, 32, 32, nt=4, nbound=6))  # sinc tables, sponge
    H.set_autotune(False)
    H.set_checkpoint_budget(nt * cells * 4)
    B = pyborn.Batch(H, [shot], (10.0, 10.0, 10.0))
    B.forward(1, nt, 0)
    traces = B.traces(0)
    B.adjoint_exact(1, nt, 0)
    image = B.image(0)
    assert np.abs(traces).max() > 0 and np.abs(image).max() > 0
    # the FP32 levels take 16 bytes per cell, the 24-bit ones 24
    leave = 128 << 20
    held = _fill(torch, leave)
    free = torch.cuda.mem_get_info()[0]
    assert 64 << 20 < free < 8 * cells
    H.set_storage("f24")
    with pytest.raises(pyborn.BornError, match="NOMEM"):
        B.forward(1, nt, 0)
    H.set_storage("f32")
    B.adjoint_exact(1, nt, 0)
    again = B.image(0)
    B.forward(1, nt, 0)
    traces2 = B.traces(0)
    del held
    torch.cuda.empty_cache()
    H.set_storage("f24")
    B.forward(1, nt, 0)
    wide = B.traces(0)
    B.close()
    H.close()
    assert np.array_equal(again, image)
    assert np.array_equal(traces2, traces)
    # one rounding of 2^-16 per step and field
    assert np.linalg.norm(wide - traces) <= 2 * nt * 2.0**-16 * np.linalg.norm(traces)
