"""Scans against the oracle, bit for bit: float and double rows in PDL's
order, short and strided rows of any type, and long integer rows cut into
chunks, at row counts and lengths around the groups, chunks and cuts."""
import numpy as np
import pytest

from pdl_amd import core as C
from oracle import pdlcpu as O
from test_gpu_parity import device, pair, rand, run_both, same, view  # noqa: F401

pytestmark = pytest.mark.gpu

OPS = ["cumusumover", "cumuprodover", "dcumusumover", "dcumuprodover"]
SHAPES = [(1, 1), (1, 15), (2, 16), (3, 17), (2, 1025), (3, 4099), (1, 30000), (1025, 33), (2500, 20), (40000, 17),
          (600, 100), (4000, 1)]


def layouts(a, t, badflag=False):
    yield "rows", pair(a, t, badflag)
    yield "columns", tuple(p.xchg(0, 1) for p in pair(np.ascontiguousarray(a.T), t, badflag))
    wide = np.repeat(a, 2, axis=1)
    yield "stepped", tuple(view(p, [("slice", (1, 2 * a.shape[1] - 1, 2), None)]) for p in pair(wide, t, badflag))


@pytest.mark.parametrize("shape", SHAPES, ids=["%dx%d" % s for s in SHAPES])
@pytest.mark.parametrize("t", [O.B, O.S, O.LL, O.F, O.D], ids=lambda t: O.TYPE_NAMES[t])
def test_scans_bit_exact(t, shape):
    rng = np.random.default_rng(50 + t)
    a = rand(t, shape, rng)
    if t >= O.F:
        a = (a / 10).astype(a.dtype)
        a.reshape(-1)[3::1001] = np.inf
        a.reshape(-1)[7::1003] = np.nan
    for name, A in layouts(a, t):
        for op in OPS:
            (o, d), = run_both(op, [A])
            same(o, d, "%s %s" % (op, name))
    a.reshape(-1)[::3] = O.default_badval(t)
    for name, A in layouts(a, t, True):
        for op in OPS[:2]:
            (o, d), = run_both(op, [A])
            same(o, d, "%s bad %s" % (op, name))


@pytest.mark.parametrize("shape", [(3, 32767), (3, 32768), (2, 65536), (1, 100003), (511, 33001), (512, 33001), (1, 1 << 21)],
                         ids=lambda s: "%dx%d" % s)
@pytest.mark.parametrize("t", [O.S, O.L, O.LL], ids=lambda t: O.TYPE_NAMES[t])
def test_long_integer_rows_bit_exact(t, shape):
    rng = np.random.default_rng(60 + t)
    a = rand(t, shape, rng)
    odd = (a | 1).astype(a.dtype)   # products stay nonzero
    for op, x in (("cumusumover", a), ("cumuprodover", odd)):
        (o, d), = run_both(op, [pair(x, t)])
        same(o, d, op)
    a.reshape(-1)[::3] = O.default_badval(t)
    (o, d), = run_both("cumusumover", [pair(a, t, True)])
    same(o, d, "cumusumover bad")


def test_in_place_and_under_capture():
    rng = np.random.default_rng(70)
    for t, shape in ((O.F, (5, 9000)), (O.L, (2, 70000))):
        a = rand(t, shape, rng)
        (o, d), = run_both("cumusumover", [pair(a, t)])
        x = C.ndarray.from_numpy(a, t)
        C._run("cumusumover", [x, x])
        assert x.numpy().tobytes() == d.numpy().tobytes()
        x, y = C.ndarray.from_numpy(a, t), C.ndarray.new_dense(t, list(shape[::-1]))
        g = C.Graph(lambda: C._run("cumusumover", [x, y]))
        for _ in range(3):
            g.launch()
            C.synchronize()
            assert y.numpy().tobytes() == d.numpy().tobytes()
            x.cumusumover()
        g.destroy()
