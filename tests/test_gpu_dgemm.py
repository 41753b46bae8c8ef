"""Double matmult on the FP64 matrix cores in the default mode, at the edges of
its tiles (32 and 64 wide), stages (16 k, the short one first) and of the cut
along t, over layouts and batches.  Entries are small whole numbers, so every
order of summation gives the exact product and nothing is tolerated; infinite
and NaN entries give the plain loop's classes."""
import numpy as np
import pytest

from pdl_amd import core as C
from oracle import pdlcpu as O

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def device():
    C.init(0)
    C.set_matmult_precision("split16")
    yield


def whole(rng, *shape):
    return rng.integers(-9, 10, shape).astype(np.float64)


LAYOUTS = {"dense": lambda m: C.ndarray.from_numpy(m, O.D),
           "transposed": lambda m: C.ndarray.from_numpy(np.ascontiguousarray(m.swapaxes(-1, -2)), O.D).xchg(0, 1),
           # every second column of a wider array, starting at an odd element
           "stepped": lambda m: C.ndarray.from_numpy(np.repeat(m, 2, axis=-1), O.D).slice((1, 2 * m.shape[-1] - 1, 2))}
SHAPES = [(8, 8, 8), (9, 15, 33), (16, 16, 16), (17, 17, 31), (32, 31, 32), (33, 32, 65), (64, 33, 64), (65, 48, 63),
          (64, 49, 96), (97, 47, 129), (20, 3000, 20), (300, 1000, 301), (1100, 64, 1030), (1030, 190, 70)]


@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "x".join(map(str, s)))
@pytest.mark.parametrize("la", list(LAYOUTS))
@pytest.mark.parametrize("lb", list(LAYOUTS))
def test_whole_numbers_exact(shape, la, lb):
    h, t, w = shape
    rng = np.random.default_rng(h + 7 * t + 31 * w)
    a, b = whole(rng, h, t), whole(rng, t, w)
    got = C.matmult(LAYOUTS[la](a), LAYOUTS[lb](b)).numpy()
    np.testing.assert_array_equal(got, a @ b)


@pytest.mark.parametrize("shape", [(3, 40, 9, 33), (70, 12, 20, 12), (5, 65, 33, 130), (2, 300, 200, 70)],
                         ids=lambda s: "x".join(map(str, s)))
@pytest.mark.parametrize("lb", list(LAYOUTS))
def test_batches_exact(shape, lb):
    n, h, t, w = shape
    rng = np.random.default_rng(n + h)
    a, b = whole(rng, n, h, t), whole(rng, n, t, w)
    np.testing.assert_array_equal(C.matmult(LAYOUTS["dense"](a), LAYOUTS[lb](b)).numpy(), a @ b)
    # one right operand for the whole batch
    np.testing.assert_array_equal(C.matmult(LAYOUTS["dense"](a), LAYOUTS[lb](b[0])).numpy(), a @ b[0])


def test_output_through_a_view_and_nonfinite_entries():
    rng = np.random.default_rng(3)
    a, b = whole(rng, 70, 45), whole(rng, 45, 90)
    out = C.ndarray.from_numpy(np.full((90, 70), 7.0), O.D)
    C.matmult(LAYOUTS["dense"](a), LAYOUTS["dense"](b), out.xchg(0, 1))
    np.testing.assert_array_equal(out.numpy().T, a @ b)
    a[3, 44], a[60, 0], b[20, 5], b[7, 89] = np.inf, np.nan, -np.inf, np.nan
    with np.errstate(invalid="ignore"):
        want = (a[:, :, None] * b[None]).sum(axis=1)
    np.testing.assert_array_equal(C.matmult(LAYOUTS["dense"](a), LAYOUTS["dense"](b)).numpy(), want)


def test_replays_of_a_cut_product():
    """the parts along t live in scratch a graph keeps; replays between eager
    products of the same shape give the eager result"""
    rng = np.random.default_rng(4)
    a, b = (LAYOUTS["dense"](whole(rng, *s)) for s in ((100, 2000), (2000, 90)))
    a2 = LAYOUTS["dense"](whole(rng, 100, 2000))
    c, ref = C.ndarray.new_dense(O.D, [90, 100]), C.ndarray.new_dense(O.D, [90, 100])
    C.matmult(a, b, ref)
    g = C.Graph(lambda: C._run("matmult", [a, b, c]))
    for _ in range(3):
        C.matmult(a2, b)
        g.launch()
        C.synchronize()
        np.testing.assert_array_equal(c.numpy(), ref.numpy())
    g.destroy()
