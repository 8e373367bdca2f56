"""Every launch shape of the steps whose form the grid decides, bit for bit.

s and r lie together or apart in the levels of the FP32 forward and of the
reference adjoint; each form is a kernel of its own for each of the 34 launch
shapes.  Each case pins one shape, checks which form ran and compares with one
fixed shape, whose results other tests hold against the CPU oracle."""
import numpy as np
import pytest

from cases import hip_prop, make_case

pytestmark = pytest.mark.gpu

REF = (1, 8, 1, 1)
# (rows per thread, wavefronts per block, cells per lane, lookahead)
SHAPES = [t + (la,) for la in (1, 2)
          for t in ((2, 4, 1), (4, 4, 1), (2, 8, 1), (2, 16, 1), (1, 8, 1), (1, 16, 1), (1, 4, 2),
                    (2, 4, 2), (1, 8, 2), (2, 8, 2), (1, 12, 2), (2, 2, 2))]
SHAPES += [(1, 4, 4, 1), (1, 2, 4, 1), (2, 2, 4, 1), (1, 8, 4, 1), (1, 1, 4, 1), (1, 3, 4, 1),
           (1, 4, 4, 2), (1, 2, 4, 2), (1, 2, 2, 1), (2, 1, 2, 1)]
_want = {}


def _same(key, run, shape, zcs):
    """run(shape, zc) against run(REF, 64), which is kept"""
    if key not in _want:
        _want[key] = run(REF, 64)
        assert all(np.abs(w).max() > 0 for w in _want[key])
    for zc in zcs:
        for got, want in zip(run(shape, zc), _want[key]):
            assert np.array_equal(got, want), (key, shape, zc)


def _device(c):
    import torch

    dev = torch.device("cuda:0")
    return (torch, torch.from_numpy(np.ascontiguousarray(c.model).ravel()).to(dev),
            torch.zeros((c.ntb, c.nrec), device=dev), dev)


@pytest.mark.parametrize("form,scatter", [("apart", 0), ("apart", 1), ("together", 1)])
@pytest.mark.parametrize("shape", SHAPES)
def test_forward(pyborn, shape, form, scatter):
    # rows of a multiple of 4 but of no tile; s levels by themselves in the
    # history of a small grid (scatter 0), in a checkpoint plan (scatter 1)
    c = make_case(124, 27, 25, nt=14, nbound=8, src_z=9, rec_z=7, seed=3, jt=3)
    torch, m, tr, _ = _device(c)

    def run(shape, zc):
        H = hip_prop(pyborn, c)
        H.transfer_receiver_func(c.rec_nx, c.rec_ny, c.rec_locs,
                                 np.zeros((c.nrec, c.ntb), np.float32))
        H.set_tuning("fwd" if scatter == 0 else "fwd_dV", *shape, zc)
        if form == "apart" and scatter == 1:
            H.set_checkpoint_budget(10 * 4 * c.nx * c.ny * c.nz)
        tr.zero_()
        torch.cuda.synchronize()
        H.dev_forward(c.jt, c.nt, m, tr, scatter, form == "apart")
        H.synchronize()
        assert H.last_levels_together[0] == (form == "together")
        H.close()
        return [tr.cpu().numpy()]

    # scatter 1 gives one result in both forms
    _same(("forward", scatter), run, shape, (3, 13))


@pytest.mark.parametrize("shape", SHAPES)
def test_source(pyborn, shape):
    c = make_case(124, 27, 25, nt=15, rand_band=4, nbound=8, src_z=9, seed=3)

    def run(shape, zc):
        H = hip_prop(pyborn, c)
        H.set_tuning("source", *shape, zc)
        p = [np.zeros(c.nx * c.ny * c.nz, np.float32) for _ in range(2)]
        H.source_prop(p[0], p[1], 1, c.nt)
        H.close()
        return p

    _same("source", run, shape, (3, 13))


@pytest.mark.parametrize("together", [False, True])
@pytest.mark.parametrize("shape", SHAPES)
def test_reference_adjoint(pyborn, shape, together):
    # 2^21 cells and 48 steps are the least of levels together
    n, nt = ((132, 133, 124), 48) if together else ((124, 27, 25), 15)
    key = ("case", together)
    if key not in _want:
        _want[key] = make_case(*n, nt=nt, rand_band=4, nbound=8, src_z=9, rec_z=7, seed=3,
                               vel_law="const")
    c = _want[key]
    torch, _, _, dev = _device(c)
    res = np.random.default_rng(7).standard_normal((c.ntb, c.nrec)).astype(np.float32)
    start = np.random.default_rng(8).standard_normal((2, c.nx * c.ny * c.nz)).astype(np.float32)

    def run(shape, zc):
        H = hip_prop(pyborn, c)
        H.transfer_receiver_func(c.rec_nx, c.rec_ny, c.rec_locs,
                                 np.zeros((c.nrec, c.ntb), np.float32))
        H.set_tuning("rtm_adjoint", *shape, zc)
        H.set_tuning("source", *REF, 64)
        t = [torch.from_numpy(a).to(dev) for a in (start[0], start[1], start[0] * 0, res)]
        torch.cuda.synchronize()
        q = [torch.zeros_like(t[0]) for _ in range(2)]
        H.dev_source_prop(1, 2, q[0], q[1])  # sets the step per sample
        H.dev_rtm_adjoint(nt, *t)
        H.synchronize()
        assert H.last_levels_together[1] == together
        H.close()
        return [a.cpu().numpy() for a in t[:3]]

    _same(("adjoint", together), run, shape, (13,) if together else (3, 13))


# 2^19 and 14 M cells bound the grids whose kept history lies beside s and r;
# with gaps in the history it is 10 M
@pytest.mark.parametrize("n,scatter,keep,gaps,together", [
    ((64, 64, 127), 0, False, False, True), ((64, 64, 127), 0, True, False, False),
    ((64, 64, 128), 0, True, False, True), ((64, 64, 128), 0, True, True, True),
    ((64, 64, 127), 1, True, False, True), ((64, 64, 127), 1, True, True, False),
    ((256, 256, 160), 0, True, False, True), ((256, 256, 160), 0, True, True, False),
    ((256, 256, 160), 1, True, True, False), ((256, 256, 216), 0, True, False, False),
    ((256, 256, 216), 1, True, False, True), ((256, 256, 216), 0, False, False, True)])
def test_form_of_the_forward(pyborn, n, scatter, keep, gaps, together):
    import torch

    c = make_case(32, 32, 32, nt=24, nbound=8)
    H = hip_prop(pyborn, c)
    H.create_space(*c.d, *n)
    H.set_autotune(False)
    cells = n[0] * n[1] * n[2]
    at = n[0] // 2 + n[0] * (n[1] // 2 + n[1] * 20)
    nt = 8
    H.transfer_source_func(np.array([at], np.int32), np.ones((1, nt + 8), np.float32))
    H.transfer_vel_func2(np.full(cells, 1e-3, np.float32))
    H.transfer_receiver_func(2, 1, np.array([at, at + 1], np.int32),
                             np.zeros((2, nt + 8), np.float32))
    if gaps:
        H.set_placement("timed", 6 * 4 * cells)
    m = torch.ones(cells, device="cuda:0")
    tr = torch.zeros((nt + 8, 2), device="cuda:0")
    torch.cuda.synchronize()
    H.dev_forward(1, nt, m, tr, scatter, keep)
    H.synchronize()
    assert H.last_levels_together[0] == together
    assert float(tr.abs().max()) > 0
    H.close()
