"""Reductions along a strided core dim, and of rows shorter than a wave,
against the oracle: numbers of outputs around the 64 a block covers, lengths
around the eight-element steps and the chunk edges, stepped and reversed
slices, bad values, and a capture without scratch."""
import numpy as np
import pytest

from pdl_amd import core as C
from oracle import pdlcpu as O
from test_gpu_parity import check_sum, device, pair, rand, run_both, same, truth_sum, view  # noqa: F401

pytestmark = pytest.mark.gpu

EXACT = ["minimum", "maximum", "minimum_ind", "maximum_ind"]
COLUMNS = [("xchg", 0, 1)]
LAYOUTS = [  # (numpy shape, view)
    ((1, 3), COLUMNS), ((7, 1), COLUMNS), ((33, 2), COLUMNS), ((70, 63), COLUMNS), ((81, 64), COLUMNS),
    ((32 * 25 + 1, 65), COLUMNS), ((10007, 3), COLUMNS), ((4099, 24), COLUMNS), ((5, 1000), COLUMNS),
    ((4, 37, 129), [("mv", 1, 0)]), ((3, 50, 5), [("mv", 2, 0)]),
    ((9, 200), [("slice", (0, 199, 2), None)]), ((3, 5000), [("slice", (4999, 0, -1), None)]),
    ((1, 20011), [("slice", (0, 20010, 3), None)]),
    ((300, 1), []), ((301, 2), []), ((17, 15), []), ((5, 33), []), ((1, 63), []), ((2000, 63), []),
]


def check(op, t, A, badval=None):
    (o, d), = run_both(op, [A])
    what = "%s %s %s" % (op, O.TYPE_NAMES[t], list(A[0].dims))
    if t >= O.F and op in ("sumover", "average"):
        truth, absum = truth_sum(A[0], op, badval=badval)
        g = A[0].gather()
        allbad = None if badval is None else (g == np.asarray(badval).astype(g.dtype)).all(axis=-1)
        check_sum(d, truth, absum, what, bad_expected=allbad)
    else:
        same(o, d, what)


@pytest.mark.parametrize("shape,v", LAYOUTS, ids=["x".join(map(str, s)) + ("-" + v[0][0] if v else "") for s, v in LAYOUTS])
@pytest.mark.parametrize("t", [O.S, O.LL, O.F, O.D], ids=lambda t: O.TYPE_NAMES[t])
def test_grid_reductions(t, shape, v):
    rng = np.random.default_rng(5 + t)
    a = rand(t, shape, rng)
    A = tuple(view(p, v) for p in pair(a, t))
    for op in ["sumover", "average"] + (["prodover"] if t < O.F else []):
        check(op, t, A)
    if t >= O.F:
        a.reshape(-1)[::5] = np.nan
        a.reshape(-1)[1::7] = np.inf
        A = tuple(view(p, v) for p in pair(a, t))
    for op in EXACT:
        check(op, t, A)
    for o, d in run_both("minmaximum", [A], nout=4):   # values alone: a row of NaN sets no bad flag on the device
        assert d.numpy().tobytes() == o.gather().tobytes(), "minmaximum"
    bv = O.default_badval(t)
    a = rand(t, shape, rng)
    a.reshape(-1)[::3] = bv
    a[..., 0] = bv
    A = tuple(view(p, v) for p in pair(a, t, True))
    for op in ["sumover", "average"] + EXACT:
        check(op, t, A, badval=bv)


def test_column_sums_under_capture():
    """a capture needs no earlier run of the op, and replays give the eager bits"""
    rng = np.random.default_rng(9)
    x = C.ndarray.from_numpy(rng.standard_normal((30011, 6)).astype(np.float32)).xchg(0, 1)
    out, ref = C.ndarray.new_dense(O.F, [6]), C.ndarray.new_dense(O.F, [6])
    g = C.Graph(lambda: C._run("minimum", [x, out]))
    C._run("minimum", [x, ref])
    for _ in range(3):
        g.launch()
        C.synchronize()
        assert out.numpy().tobytes() == ref.numpy().tobytes()
        x.sumover()
    g.destroy()
