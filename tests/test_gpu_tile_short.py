"""Float products of few k, up to and past the half stage of 16 that has a
kernel form of its own: every tile shape and layout, batches, whole numbers
exactly, infinities and NaN as in the plain loop, and the error of normal
data, which is that of sums of 8 k joined (2^-23 of the norm at 17 k)."""
import numpy as np
import pytest

from pdl_amd import core as C
from test_gpu_dgemm import device, whole  # noqa: F401
from test_gpu_tile_f32 import LAYOUTS

pytestmark = pytest.mark.gpu

TS = [8, 9, 12, 15, 16, 17, 32]
SIDES = [(64, 64), (33, 31), (40, 70), (200, 33), (8, 300), (129, 65)]


@pytest.mark.parametrize("t", TS)
@pytest.mark.parametrize("la", list(LAYOUTS))
@pytest.mark.parametrize("lb", list(LAYOUTS))
def test_whole_numbers_exact(t, la, lb):
    for h, w in SIDES:
        rng = np.random.default_rng(h + 7 * t + 31 * w)
        a, b = whole(rng, h, t), whole(rng, t, w)
        np.testing.assert_array_equal(C.matmult(LAYOUTS[la](a), LAYOUTS[lb](b)).numpy(), a @ b)
        a, b = whole(rng, 5, h, t), whole(rng, 5, t, w)
        np.testing.assert_array_equal(C.matmult(LAYOUTS[la](a), LAYOUTS[lb](b)).numpy(), a @ b)


@pytest.mark.parametrize("t", TS)
def test_nonfinite_entries_and_error(t):
    rng = np.random.default_rng(t)
    a, b = whole(rng, 70, t), whole(rng, t, 90)
    a[3, t - 1], a[60, 0], b[t // 2, 5], b[7, 89] = np.inf, np.nan, -np.inf, np.nan
    with np.errstate(invalid="ignore"):
        want = (a[:, :, None] * b[None]).sum(axis=1)
    np.testing.assert_array_equal(C.matmult(LAYOUTS["dense"](a), LAYOUTS["dense"](b)).numpy(), want)
    a, b = rng.standard_normal((300, t)).astype(np.float32), rng.standard_normal((t, 200)).astype(np.float32)
    truth = a.astype(np.float64) @ b.astype(np.float64)
    d = C.matmult(LAYOUTS["dense"](a), LAYOUTS["dense"](b)).numpy() - truth
    assert np.linalg.norm(d) <= 2.0 ** -23 * np.linalg.norm(truth)
