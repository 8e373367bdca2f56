"""Forms of the step kernels that a rule on sizes chooses.

Every form evaluates a cell with the same roundings, so results are compared
bit for bit where two forms can run the same problem, and with the CPU oracle
at its parity bound (1e-4 relative l2, FP32) where only one can: the launch
shapes of four cells per lane and of 32x8 tiles, s and r stored together or
apart, receiver values carried over several windows, and results copied out
through the pinned ring (from 4 MB)."""
import numpy as np
import pytest

from cases import hip_prop, make_case, oracle_prop, rel_l2

pytestmark = pytest.mark.gpu

PARITY = 1e-4
REF = (1, 8, 1, 1)
# (rows per thread, wavefronts per block, cells per lane, lookahead)
SHAPES = [(1, 4, 4, 1), (1, 2, 4, 1), (2, 2, 4, 1), (1, 8, 4, 1), (1, 1, 4, 1), (1, 3, 4, 1),
          (1, 4, 4, 2), (1, 2, 4, 2), (1, 2, 2, 1), (2, 1, 2, 1)]


def _pair(H, c, w, scatter, keep):
    """Born data and exact-adjoint image on device tensors."""
    import torch

    dev = torch.device("cuda:0")
    m = torch.from_numpy(np.ascontiguousarray(c.model).ravel()).to(dev)
    tr = torch.zeros((c.ntb, c.nrec), device=dev)
    img = torch.zeros(c.nx * c.ny * c.nz, device=dev)
    res = torch.from_numpy(np.ascontiguousarray(w.T)).to(dev)
    torch.cuda.synchronize()
    H.dev_forward(c.jt, c.nt, m, tr, scatter, keep)
    H.dev_adjoint_exact(c.jt, c.nt, res, img, scatter)
    H.synchronize()
    return tr.cpu().numpy(), img.cpu().numpy()


def _prop(pyborn, c, storage="f32"):
    H = hip_prop(pyborn, c)
    H.set_storage(storage)
    H.transfer_receiver_func(c.rec_nx, c.rec_ny, c.rec_locs,
                             np.zeros((c.nrec, c.ntb), np.float32))
    return H


@pytest.mark.parametrize("storage", ["f32", "f16", "f24"])
@pytest.mark.parametrize("shape", SHAPES)
def test_shapes_give_the_same_bits(pyborn, shape, storage):
    # rows of a multiple of 4 but of no tile; chunks of one plane, of an odd
    # number and longer than the domain
    c = make_case(124, 27, 25, nt=14, nbound=8, src_z=9, rec_z=7, seed=3, jt=3)
    w = np.random.default_rng(2).standard_normal((c.nrec, c.ntb)).astype(np.float32)
    sfx = "" if storage == "f32" else "_" + storage
    kinds = [k + sfx for k in ("fwd", "background", "adjoint_state")]

    def run(shape, zc, keep):
        H = _prop(pyborn, c, storage)
        for k in kinds:
            H.set_tuning(k, *shape, zc)
        out = _pair(H, c, w, 0, keep)
        H.close()
        return out

    want = run(REF, 64, False)
    assert np.abs(want[0]).max() > 0 and np.abs(want[1]).max() > 0
    for zc, keep in ((1, False), (3, True), (64, False)):
        got = run(shape, zc, keep)
        assert np.array_equal(got[0], want[0]) and np.array_equal(got[1], want[1]), (shape, zc)


@pytest.mark.parametrize("scatter", [0, 1])
@pytest.mark.parametrize("n", [(64, 64, 127), (64, 64, 128), (97, 75, 74)])
def test_levels_together_and_apart(pyborn, n, scatter):
    # 2^19 cells are the least of a kept history whose s levels stay with r.
    # Without a history s and r are together, with a checkpoint plan apart;
    # with gaps in the history (short windows) the size decides
    c = make_case(*n, nt=24, nbound=8, src_z=9, rec_z=7, seed=5)
    w = np.random.default_rng(3).standard_normal((c.nrec, c.ntb)).astype(np.float32)
    out = []
    F = 4 * c.nx * c.ny * c.nz
    for form in ("no history", "history", "gaps", "checkpoints"):
        H = _prop(pyborn, c)
        if form == "gaps":
            H.set_placement("timed", 10 * F)
        if form == "checkpoints":
            H.set_checkpoint_budget(16 * F)
        out.append(_pair(H, c, w, scatter, form != "no history"))
        if form == "checkpoints":
            assert H.last_checkpoint_plan()[0] >= 2
        H.close()
    for got in out[1:]:
        assert np.array_equal(got[0], out[0][0]) and np.array_equal(got[1], out[0][1])
    assert np.abs(out[0][0]).max() > 0 and np.abs(out[0][1]).max() > 0


# 2^21 cells and 48 steps are the least of a reference adjoint whose levels
# are together; the last grid is odd in every direction
@pytest.mark.parametrize("n,nt", [((128, 128, 128), 48), ((128, 128, 128), 47),
                                  ((128, 128, 127), 48), ((131, 127, 129), 49)])
def test_reference_adjoint_levels(pyborn, n, nt):
    c = make_case(*n, nt=nt, rand_band=8, nbound=10)
    traces = np.random.default_rng(7).standard_normal((c.nrec, c.ntb)).astype(np.float32)
    P = oracle_prop(c)
    P.transfer_receiver_func(c.rec_locs, traces.copy())
    H = hip_prop(pyborn, c)
    H.transfer_receiver_func(c.rec_nx, c.rec_ny, c.rec_locs, traces.copy())
    got = []
    for X in (P, H):
        a = [np.zeros(c.nx * c.ny * c.nz, np.float32) for _ in range(3)]
        X.source_prop(a[0], a[1], 1, nt)
        before = [np.linalg.norm(x.astype(np.float64)) for x in a]
        X.rtm_adjoint(a[1], a[0], a[2], nt)
        got.append(a)
    H.close()
    # An even nt takes the state back to rest, to the rounding of the field it
    # came from (2.4e-7 of its norm in the oracle): errors of the two states are
    # relative to that field, the image's to the image.
    for o, h, b in zip(*got, before):
        assert np.abs(o).max() > 0
        err = np.linalg.norm(h.astype(np.float64) - o)
        assert err <= PARITY * max(np.linalg.norm(o.astype(np.float64)), b)


@pytest.mark.parametrize("jt", [1, 4])
def test_receiver_windows(pyborn, jt):
    # 13,000 receivers, 700 steps: more receiver values than the 32 MB of a
    # window; every seventh receiver shares its cell with another
    c = make_case(142, 112, 20, nt=700, rec_step=1, nbound=6, src_z=8, jt=jt)
    c.rec_locs[3::7] = c.rec_locs[1::7][: len(c.rec_locs[3::7])]
    assert c.nrec * c.nt * 4 > 32 << 20
    w = np.random.default_rng(9).standard_normal((c.nrec, c.ntb)).astype(np.float32)
    P = oracle_prop(c)
    rec = np.zeros((c.nrec, c.ntb), np.float32)
    P.transfer_receiver_func(c.rec_locs, rec)
    P.rtm_forward(c.jt, c.model, c.nt)
    H = hip_prop(pyborn, c)
    d = np.zeros((c.nrec, c.ntb), np.float32)
    H.transfer_receiver_func(c.rec_nx, c.rec_ny, c.rec_locs, d)
    H.forward_scatter(c.jt, c.model, d, c.nt, 0)
    assert np.abs(rec).max() > 0 and rel_l2(d, rec) <= PARITY
    img = np.zeros(c.nx * c.ny * c.nz, np.float32)
    H.adjoint_exact(c.jt, w, img, c.nt, scatter=0)
    # <F m, w> = <m, F^T w>: FP32 errors of 3e-6 of each value, uncorrelated,
    # sum to 3e-6 of these magnitudes; a window in the wrong place to about 1
    d64, w64 = d.astype(np.float64).ravel(), w.astype(np.float64).ravel()
    m64, i64 = c.model.astype(np.float64).ravel(), img.astype(np.float64)
    scale = sum(np.linalg.norm(x) * np.linalg.norm(y) / np.sqrt(x.size)
                for x, y in ((d64, w64), (m64, i64)))
    assert abs(np.dot(d64, w64) - np.dot(m64, i64)) <= PARITY * scale
    B = pyborn.Batch(H, [{"nx": c.nx, "ny": c.ny, "nz": c.nz, "vel": c.V2, "model": c.model,
                          "src_locs": c.src_locs, "src_vals": c.src_vals, "rec_nx": c.rec_nx,
                          "rec_ny": c.rec_ny, "rec_locs": c.rec_locs}], c.d)
    B.forward(c.jt, c.nt, 0)
    assert np.array_equal(B.traces(0), d)
    B.set_traces(0, w)
    B.adjoint_exact(c.jt, c.nt, 0)
    assert np.array_equal(B.image(0), img)
    B.close()
    H.close()
