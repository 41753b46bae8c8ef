"""Float matmult on the FP32 matrix cores in the default mode: the shapes,
layouts and batches of the double tests (small whole numbers, exact in any
order), the side at which the kernels hand over to each other, and the error
of normal data, which is at most a few roundings per 32 k: 2^-22 of the
product's norm covers any of these sizes."""
import numpy as np
import pytest

from pdl_amd import core as C
from oracle import pdlcpu as O
from test_gpu_dgemm import SHAPES, device, whole  # noqa: F401

pytestmark = pytest.mark.gpu

LAYOUTS = {"dense": lambda m: C.ndarray.from_numpy(m, O.F),
           "transposed": lambda m: C.ndarray.from_numpy(np.ascontiguousarray(m.swapaxes(-1, -2)), O.F).xchg(0, 1),
           "stepped": lambda m: C.ndarray.from_numpy(np.repeat(m, 2, axis=-1), O.F).slice((1, 2 * m.shape[-1] - 1, 2))}


@pytest.mark.parametrize("shape", SHAPES + [(40, 96, 70), (40, 97, 70), (32, 33, 33), (33, 33, 33), (64, 64, 65)],
                         ids=lambda s: "x".join(map(str, s)))
@pytest.mark.parametrize("la", list(LAYOUTS))
@pytest.mark.parametrize("lb", list(LAYOUTS))
def test_whole_numbers_exact(shape, la, lb):
    h, t, w = shape
    rng = np.random.default_rng(h + 7 * t + 31 * w)
    a, b = whole(rng, h, t), whole(rng, t, w)
    got = C.matmult(LAYOUTS[la](a), LAYOUTS[lb](b)).numpy()
    np.testing.assert_array_equal(got, (a @ b).astype(np.float32))


@pytest.mark.parametrize("shape", [(3, 40, 9, 33), (70, 12, 20, 12), (5, 65, 33, 130), (2, 300, 200, 70), (9, 32, 64, 64)],
                         ids=lambda s: "x".join(map(str, s)))
@pytest.mark.parametrize("lb", list(LAYOUTS))
def test_batches_exact(shape, lb):
    n, h, t, w = shape
    rng = np.random.default_rng(n + h)
    a, b = whole(rng, n, h, t), whole(rng, n, t, w)
    np.testing.assert_array_equal(C.matmult(LAYOUTS["dense"](a), LAYOUTS[lb](b)).numpy(), a @ b)
    np.testing.assert_array_equal(C.matmult(LAYOUTS["dense"](a), LAYOUTS[lb](b[0])).numpy(), a @ b[0])


@pytest.mark.parametrize("shape", [(70, 16, 80), (90, 96, 90), (300, 700, 200), (100, 5000, 60), (1000, 1000, 1000)],
                         ids=lambda s: "x".join(map(str, s)))
def test_error_of_normal_data(shape):
    h, t, w = shape
    rng = np.random.default_rng(h + t)
    a, b = rng.standard_normal((h, t)).astype(np.float32), rng.standard_normal((t, w)).astype(np.float32)
    d = C.matmult(LAYOUTS["dense"](a), LAYOUTS["dense"](b)).numpy().astype(np.float64)
    truth = a.astype(np.float64) @ b.astype(np.float64)
    assert np.linalg.norm(d - truth) <= 2.0 ** -22 * np.linalg.norm(truth)
