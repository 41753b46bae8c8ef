"""Reductions and scans at the lines between their kernels: rows of up to 7
elements and 16 bytes, 64 bytes and more; columns of fewer than 16 elements
where their number fills the chip; integer scans of long rows where they are
cut and where not; scans of up to 16 elements."""
import numpy as np
import pytest

from oracle import pdlcpu as O
from test_gpu_parity import device, pair, rand, run_both, same, view  # noqa: F401
from test_gpu_reduce_grid import check

pytestmark = pytest.mark.gpu


def both_ways(t, a, v):
    bv = O.default_badval(t)
    A = tuple(view(p, v) for p in pair(a, t))
    for op in ("sumover", "average", "minimum", "maximum_ind") + (("prodover",) if t < O.F else ()):
        check(op, t, A)
    a.reshape(-1)[::3] = bv
    a[..., 0] = bv
    A = tuple(view(p, v) for p in pair(a, t, True))
    for op in ("sumover", "minimum"):
        check(op, t, A, badval=bv)


@pytest.mark.parametrize("n", [1, 2, 4, 7, 8, 9, 15, 16, 17, 31, 32, 33, 63])
@pytest.mark.parametrize("t", [O.B, O.S, O.F, O.D], ids=lambda t: O.TYPE_NAMES[t])
def test_short_rows(t, n):
    rng = np.random.default_rng(n)
    for rows in (3, 1031):
        both_ways(t, rand(t, (rows, n), rng), [])


WAVES = [(256, 8200), (257, 8200), (1280, 2048), (1281, 2048), (1600, 6400), (1601, 6400), (300, 102401), (640, 102400), (641, 102400),
         (4095, 19200), (4096, 19200), (4095, 19199), (40, 2047)]


# the longest as bytes only: the same path, and the oracle's pass over them is long
@pytest.mark.parametrize("t,rows,n", [(t, r, n) for t in (O.B, O.F) for r, n in WAVES if t == O.B or r * n <= 2 ** 25],
                         ids=lambda s: str(s))
def test_waves_per_row(t, rows, n):
    rng = np.random.default_rng(rows)
    A = pair(rand(t, (rows, n), rng), t)
    for op in ("sumover", "maximum_ind"):
        check(op, t, A)


@pytest.mark.parametrize("n", [1, 4, 15, 16, 17])
@pytest.mark.parametrize("cols", [262143, 262144, 262147])
@pytest.mark.parametrize("t", [O.S, O.D], ids=lambda t: O.TYPE_NAMES[t])
def test_many_short_columns(t, n, cols):
    rng = np.random.default_rng(n + cols)
    both_ways(t, rand(t, (n, cols), rng), [("xchg", 0, 1)])


@pytest.mark.parametrize("rows", [255, 256])
@pytest.mark.parametrize("t", [O.L, O.LL], ids=lambda t: O.TYPE_NAMES[t])
def test_integer_scans_cut_and_whole(t, rows):
    rng = np.random.default_rng(rows)
    a = rand(t, (rows, 33001), rng)
    (o, d), = run_both("cumusumover", [pair(a, t)])
    same(o, d, "cumusumover")
    a.reshape(-1)[::3] = O.default_badval(t)
    (o, d), = run_both("cumusumover", [pair(a, t, True)])
    same(o, d, "cumusumover bad")


@pytest.mark.parametrize("n", [1, 7, 15, 16, 17, 32, 33])
@pytest.mark.parametrize("rows", [600, 1024, 40001])
@pytest.mark.parametrize("t", [O.B, O.L, O.F, O.D], ids=lambda t: O.TYPE_NAMES[t])
def test_short_scans(t, n, rows):
    rng = np.random.default_rng(n + rows)
    a = rand(t, (rows, n), rng)
    for A in (pair(a, t), tuple(p.xchg(0, 1) for p in pair(np.ascontiguousarray(a.T), t))):
        for op in ("cumusumover", "dcumusumover"):
            (o, d), = run_both(op, [A])
            same(o, d, op)
    a.reshape(-1)[::3] = O.default_badval(t)
    (o, d), = run_both("cumusumover", [pair(a, t, True)])
    same(o, d, "cumusumover bad")
