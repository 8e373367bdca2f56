"""Steps of grids past the memory-side cache, whose loads and stores take the
non-temporal hint: the bits of the kernels that do without it, bit for bit.

FP32 with s and r together from 330 MB of levels, velocity and model (440 MB
with the dV term), against s and r apart; the narrow adjoints from 512 MB,
against a batch of the one shot."""
import numpy as np
import pytest

from cases import hip_prop, make_case

pytestmark = pytest.mark.gpu

SHAPES = [(2, 4, 1, 1), (1, 8, 2, 2), (1, 2, 4, 1)]
_data = {}


def _problem(n):
    if n not in _data:
        _data.clear()
        cells = n[0] * n[1] * n[2]
        rng = np.random.default_rng(11)
        _data[n] = (rng.uniform(1.5e-3, 4.5e-3, cells).astype(np.float32),
                    rng.standard_normal(cells, dtype=np.float32))
    return _data[n]


def _prop(pyborn, n, nt, storage, shape, kinds):
    vel, model = _problem(n)
    at = n[0] // 2 + n[0] * (n[1] // 2 + n[1] * 40)
    shot = {"nx": n[0], "ny": n[1], "nz": n[2], "vel": vel, "model": model,
            "src_locs": np.array([at], np.int32),
            "src_vals": np.ones((1, nt + 8), np.float32), "rec_nx": 6, "rec_ny": 1,
            "rec_locs": np.arange(at - 2, at + 4, dtype=np.int32)}
    H = hip_prop(pyborn, make_case(32, 32, 32, nt=4, nbound=6))  # sinc tables, sponge
    H.create_space(10.0, 10.0, 10.0, *n)
    H.set_autotune(False)
    H.set_storage(storage)
    for k in kinds:
        H.set_tuning(k, *shape, 29)
    H.transfer_source_func(shot["src_locs"], shot["src_vals"])
    H.transfer_vel_func2(vel)
    H.transfer_receiver_func(6, 1, shot["rec_locs"], np.zeros((6, nt + 8), np.float32))
    return H, shot


@pytest.mark.parametrize("shape", SHAPES)
@pytest.mark.parametrize("n,scatter", [((256, 256, 216), 0), ((272, 260, 264), 1)])
def test_fp32_forward(pyborn, n, scatter, shape):
    import torch

    nt = 6
    cells = n[0] * n[1] * n[2]
    assert 24 * cells > (330e6 if scatter == 0 else 440e6)
    dev = torch.device("cuda:0")
    m = torch.from_numpy(_problem(n)[1]).to(dev)
    out = []
    for together in (True, False):
        H, _ = _prop(pyborn, n, nt, "f32", shape, ["fwd" if scatter == 0 else "fwd_dV"])
        if not together and scatter == 1:
            H.set_checkpoint_budget(5 * 4 * cells)
        tr = torch.zeros((nt + 8, 6), device=dev)
        torch.cuda.synchronize()
        # kept, scatter 0: s in the history; scatter 1: its own history or a plan
        H.dev_forward(1, nt, m, tr, scatter, scatter == 1 or not together)
        H.synchronize()
        assert H.last_levels_together[0] == together
        img = torch.zeros(cells, device=dev)
        if scatter == 1:  # the scatter operands that the forward left
            H.dev_adjoint_exact(1, nt, tr, img, scatter)
            H.synchronize()
            assert H.last_background_sweep() == 0
        out.append((tr.cpu().numpy(), img.cpu().numpy()))
        H.close()
    assert np.abs(out[0][0]).max() > 0
    for a, b in zip(*out):
        assert np.array_equal(a, b)


@pytest.mark.parametrize("shape", SHAPES)
@pytest.mark.parametrize("storage,scatter", [("f24", 0), ("f24", 1), ("f16", 0), ("f16", 1)])
def test_narrow_pair(pyborn, storage, scatter, shape):
    import torch

    n, nt = (352, 352, 352), 4
    cells = n[0] * n[1] * n[2]
    esz = {"f16": 2, "f24": 3}[storage]
    assert cells * (2 * esz + 8) > 512e6
    sc = "" if scatter == 0 else "_dV"
    kinds = [k + "_" + storage for k in ("fwd" + sc, "background" + sc, "adjoint_state")]
    H, shot = _prop(pyborn, n, nt, storage, shape, kinds)
    dev = torch.device("cuda:0")
    m = torch.from_numpy(shot["model"]).to(dev)
    tr = torch.zeros((nt + 8, 6), device=dev)
    img = torch.zeros(cells, device=dev)
    torch.cuda.synchronize()
    H.dev_forward(1, nt, m, tr, scatter, False)
    H.dev_adjoint_exact(1, nt, tr, img, scatter)
    H.synchronize()
    assert H.last_background_sweep() == nt
    if scatter not in _want.setdefault(storage, {}):
        B = pyborn.Batch(H, [shot], (10.0, 10.0, 10.0))
        B.forward(1, nt, scatter)
        B.adjoint_exact(1, nt, scatter)
        _want[storage][scatter] = (B.traces(0).T.copy(), B.image(0))
        B.close()
    H.close()
    want = _want[storage][scatter]
    assert np.abs(want[0]).max() > 0 and np.abs(want[1]).max() > 0
    assert np.array_equal(tr.cpu().numpy(), want[0])
    assert np.array_equal(img.cpu().numpy(), want[1])


_want = {}
