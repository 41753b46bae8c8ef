"""Reductions of unit-stride rows against the oracle at the edges of their
dispatch: rows starting at every offset from a 16-byte boundary, lengths
around the vectors, the waves per row (1, 4, 16) and the chunks of the split."""
import numpy as np
import pytest

from pdl_amd import core as C  # noqa: F401
from oracle import pdlcpu as O
from test_gpu_parity import device, pair, rand, view  # noqa: F401
from test_gpu_reduce_grid import check

pytestmark = pytest.mark.gpu

SHAPES = [  # (rows, length): the chosen number of waves depends on bytes per row and on rows
    (5, 64), (3, 65), (4097, 67), (4095, 1031), (1023, 4099), (1024, 2049), (1025, 2047),
    (2, 8191), (3, 16385), (7, 65537), (1, 131071), (1, 524309), (511, 66001), (512, 65999),
]


@pytest.mark.parametrize("shape", SHAPES, ids=["%dx%d" % s for s in SHAPES])
@pytest.mark.parametrize("t", [O.B, O.S, O.L, O.F, O.D], ids=lambda t: O.TYPE_NAMES[t])
def test_row_reductions(t, shape):
    if shape[0] * shape[1] > 2 ** 24 and t not in (O.B, O.F):
        pytest.skip("the same path as the other types; the oracle's pass over it is long")
    rng = np.random.default_rng(8 + t)
    a = rand(t, shape, rng)
    if t >= O.F:
        a.reshape(-1)[::101] = np.nan
    A = pair(a, t)
    for op in ["minimum", "maximum_ind"]:
        check(op, t, A)
    a = rand(t, shape, rng)
    check("sumover", t, pair(a, t))
    bv = O.default_badval(t)
    a.reshape(-1)[::3] = bv
    a[0] = bv
    check("average", t, pair(a, t, True), badval=bv)


@pytest.mark.parametrize("t", [O.B, O.S, O.L, O.D], ids=lambda t: O.TYPE_NAMES[t])
def test_rows_at_every_offset(t):
    rng = np.random.default_rng(80 + t)
    a = rand(t, (6, 3000), rng)
    for lo in range(0, 17):
        for hi in (2999, 2999 - lo, lo + 63, lo + 79):
            A = tuple(view(p, [("slice", (lo, hi, 1), None)]) for p in pair(a, t))
            for op in ["sumover", "minimum_ind"]:
                check(op, t, A)
