"""Bad.pd's elementwise ops on contiguous operands, against the oracle: counts
around the vectors and the blocks' steps, ranges that start on and off a
16-byte boundary, a mask per element and one for all."""
import numpy as np
import pytest

from pdl_amd import core as C  # noqa: F401
from oracle import pdlcpu as O
from test_gpu_ufunc_bad import NAMES, device, pair, rand, run_both, same, view  # noqa: F401

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 7, 8, 17, 2049, 4096, 8191, 70003])
@pytest.mark.parametrize("t", [O.B, O.S, O.L, O.F, O.D], ids=lambda t: NAMES[t])
def test_flat_bad_ops(t, n):
    rng = np.random.default_rng(11 + t)
    a = rand(t, (n + 16,), rng)
    bv = O.default_badval(t)
    a[::5] = bv
    mask = (rng.random(n + 16) < 0.3).astype(np.int32)
    for lo in (0, 16, 3):
        cut = [("slice", (lo, lo + n - 1, 1))]
        A = tuple(view(p, cut) for p in pair(a, t, True))
        G = tuple(view(p, cut) for p in pair(a, t))
        M = tuple(view(p, cut) for p in pair(mask, O.L))
        for op in ("isbad", "isgood"):
            for src in (A, G):
                (o, d), = run_both(op, [src])
                same(o, d, op)
        for mk in (M, pair(np.array(1, np.int32), O.L)):
            (o, d), = run_both("setbadif", [A, mk])
            same(o, d, "setbadif")
        for op, v in (("setvaltobad", float(a[lo])), ("setbadtoval", 3.0)):
            (o, d), = run_both(op, [A], dpar=v)
            same(o, d, op)
        if t >= O.F:
            x = a.copy()
            x[lo + n - 1] = np.nan
            X = tuple(view(p, cut) for p in pair(x, t))
            for op in ("setnantobad", "setinftobad"):
                (o, d), = run_both(op, [X])
                same(o, d, op)
