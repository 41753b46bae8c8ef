"""pdlhip_run_reduce_noalloc over strided and short rows: the bits of the
allocating entry, on doubles and floats that cancel (another order of
summation shows) and on whole numbers, at numbers of outputs around the 64 a
block covers and rows long enough to be cut."""
import numpy as np
import pytest

from pdl_amd import core as C
from test_zz_no_alloc import device, noalloc  # noqa: F401

pytestmark = pytest.mark.gpu

SHAPES = [(1000003, 1), (1000003, 24), (200001, 63), (100001, 64), (100001, 65), (20003, 1000), (4099, 16384),
          (70, 300000), (31, 5)]


def cancelling(rng, rows, cols, dt):
    span = 30 if dt == np.float64 else 12
    x = rng.standard_normal((rows // 2, cols)) * 10.0 ** rng.uniform(0, span, (rows // 2, cols))
    x = np.concatenate([x, -x, rng.standard_normal((rows - rows // 2 * 2, cols))]).astype(dt)
    return x[rng.permutation(rows)]


def same(op, x):
    ref = C.ndarray()
    C._run(op, [x, ref])
    out = C.ndarray.new_dense(ref.dtype, ref.dims)
    noalloc(op, x, out)
    assert out.numpy().tobytes() == ref.numpy().tobytes(), (op, x.dims)


@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "%dx%d" % s)
@pytest.mark.parametrize("dt", [np.float64, np.float32, np.int16], ids=lambda d: np.dtype(d).name)
def test_columns(shape, dt):
    rng = np.random.default_rng(shape[1])
    if dt == np.int16:
        a = rng.integers(-30000, 30000, shape).astype(dt)
    else:
        a = cancelling(rng, *shape, dt)
    x = C.ndarray.from_numpy(a).xchg(0, 1)
    for op in ("sumover", "average", "minimum", "maximum_ind"):
        same(op, x)


@pytest.mark.parametrize("n", [300001, 3000001])
def test_stepped_rows(n):
    rng = np.random.default_rng(n)
    x = C.ndarray.from_numpy(cancelling(rng, n, 1, np.float64).reshape(1, n)).slice((0, n - 1, 3), None)
    for op in ("sumover", "daverage", "maximum"):
        same(op, x)
