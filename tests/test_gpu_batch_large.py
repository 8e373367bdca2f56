"""A batch of more than 200 million cells, whose z chunks are all marched up:
each shot gives the bits of a small batch, whose chunks are turned round."""
import numpy as np
import pytest

from cases import hip_prop, make_case

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("storage", ["f32", "f24"])
def test_shots_of_a_large_batch(pyborn, storage):
    n, nt, shots = 256, 5, 12
    assert shots * n**3 > 200e6 > (shots - 1) * n**3
    rng = np.random.default_rng(6)
    vel = rng.uniform(1.5, 4.5, n**3).astype(np.float32) * np.float32(1e-3)
    model = rng.standard_normal(n**3).astype(np.float32)

    def shot(k):
        # sources next to chunk edges and in the middle of chunks
        at = 100 + 5 * k + n * (120 + n * (30 + 11 * k))
        return {"nx": n, "ny": n, "nz": n, "vel": vel, "model": model,
                "src_locs": np.array([at], np.int32),
                "src_vals": np.full((1, nt + 8), 1 + k, np.float32), "rec_nx": 6, "rec_ny": 1,
                "rec_locs": np.arange(at - 2, at + 4, dtype=np.int32)}

    H = hip_prop(pyborn, make_case(32, 32, 32, nt=4, nbound=6))  # sinc tables, sponge
    H.set_autotune(False)
    H.set_storage(storage)
    H.set_zchunk(31)
    out = []
    for ks in (range(shots), (0, shots - 1)):
        B = pyborn.Batch(H, [shot(k) for k in ks], (10.0, 10.0, 10.0))
        B.forward(1, nt, 0)
        B.adjoint_exact(1, nt, 0)
        out.append([(B.traces(s), B.image(s)) for s in (0, len(ks) - 1)])
        B.close()
    H.close()
    for got, want in zip(*out):
        for g, w in zip(got, want):
            assert np.abs(w).max() > 0
            assert np.array_equal(g, w)
