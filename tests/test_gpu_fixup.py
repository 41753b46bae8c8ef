"""Outputs of a large float product that come from PDL's loop because FP16
halves lose too much of their rows: one, two, five and many of them in a row,
at inner dimensions around the recompute's steps, equal to the PDL-order mode
bit for bit."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


# (beyond 3e10 operations the split runs whatever the tuner measures)
@pytest.mark.parametrize("t,h,w", [(300, 8192, 7000), (1000, 4160, 4160), (1025, 4096, 4096), (4096, 2100, 2048),
                                   (4100, 2048, 2048), (9000, 1400, 1400)])
def test_marked_outputs_follow_the_loop(t, h, w):
    from pdl_amd import core as C
    C.init(0)
    rng = np.random.default_rng(t)
    a = rng.standard_normal((h, t)).astype(np.float32)
    b = rng.standard_normal((t, w)).astype(np.float32)
    marked = [(3, [5]), (7, [0, w - 1]), (50, [11, 12, 13, 14, 300]), (h - 1, list(range(400, 700)))]
    for i, (r, cols) in enumerate(marked):
        big, small = 4 * i, t - 1 - 4 * i
        a[r] *= np.float32(1e-7)
        a[r, big] = 1e6
        b[big, cols] = 1e-9
        b[small, cols] = 1e7
    x, y = C.ndarray.from_numpy(a, C.L.F), C.ndarray.from_numpy(b, C.L.F)
    try:
        C.set_matmult_precision("pdlorder")
        want = C.matmult(x, y).numpy()
    finally:
        C.set_matmult_precision("split16")
    got = C.matmult(x, y).numpy()
    for r, cols in marked:
        assert np.array_equal(got[r, cols], want[r, cols]), (r, got[r, cols][:4], want[r, cols][:4])
