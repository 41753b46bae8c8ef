"""An op that runs in the middle of another on the same thread (a signal
handler, a finalizer called by the garbage collector, an operand's own code)
leaves the outer call's arguments and results alone.  Dry runs: the planner
gives output types and dims without a GPU."""
import gc
import signal
import time

import pytest

from pdl_amd import _lib as L
from pdl_amd import core as C


@pytest.fixture(autouse=True)
def plan_only():
    C.set_plan_only(True)
    yield
    C.set_plan_only(False)


def dense(t, dims):
    return C.ndarray.new_dense(t, dims)


def inner():
    """another op, of other types, dims and number of ndarrays"""
    a = dense(L.D, [7, 5, 3])
    b = C.ndarray()
    C._run("sumover", [a, b])
    assert (b.dtype, b.dims) == (L.D, [5, 3])
    c = C.ndarray()
    C._run("mult", [a, a, c])
    assert (c.dtype, c.dims) == (L.D, [7, 5, 3])


def outer():
    a, b, c = dense(L.F, [4, 6]), dense(L.F, [4, 1]), C.ndarray()
    C._run("plus", [a, b, c])
    assert (c.dtype, c.dims) == (L.F, [4, 6])


class Offset:
    """a zero that runs code when it is taken as an integer"""
    def __init__(self, f):
        self.f = f

    def __index__(self):
        self.f()
        return 0


@pytest.mark.parametrize("which", [0, 1, 2])
def test_op_while_operands_are_packed(which):
    pdls = [dense(L.F, [4, 6]), dense(L.F, [4, 1]), dense(L.F, [4, 6])]
    pdls[which].offs = Offset(inner)
    if which < 2:
        pdls[2] = C.ndarray()
    C._run("plus", pdls)
    assert (pdls[2].dtype, pdls[2].dims) == (L.F, [4, 6])


def test_op_inside_a_nested_op():
    """two levels deep, and the thread's block is whole afterwards"""
    mid = dense(L.S, [3])
    mid.offs = Offset(inner)

    def level():
        r = C.ndarray()
        C._run("sumover", [mid, r])
        assert (r.dtype, r.dims) == (L.L, [])

    a, c = dense(L.F, [4, 6]), C.ndarray()
    a.offs = Offset(level)
    C._run("plus", [a, a, c])
    assert (c.dtype, c.dims) == (L.F, [4, 6])
    outer()


def test_op_after_a_refused_one():
    a, b = dense(L.F, [4]), dense(L.F, [5])
    for _ in range(2):
        with pytest.raises(L.PDLError):
            C._run("plus", [a, b, C.ndarray()])
        outer()


def test_ops_in_a_signal_handler():
    ran = [0]

    def handler(sig, frame):
        ran[0] += 1
        inner()
        signal.setitimer(signal.ITIMER_REAL, 1e-4)   # (armed here, so that handlers do not pile up)

    old = signal.signal(signal.SIGALRM, handler)
    signal.setitimer(signal.ITIMER_REAL, 1e-4)
    try:
        end = time.monotonic() + 1.0
        while time.monotonic() < end:
            outer()
    finally:
        signal.setitimer(signal.ITIMER_REAL, 0)
        signal.signal(signal.SIGALRM, old)
    assert ran[0] > 20


@pytest.mark.parametrize("threshold", [5, 11, 13, 17])
def test_ops_in_finalizers(threshold):
    ran = [0]

    class Cycle:
        def __init__(self):
            self.me = self

        def __del__(self):
            ran[0] += 1
            inner()

    old = gc.get_threshold()
    gc.set_threshold(threshold)
    try:
        for _ in range(2000):
            Cycle()
            outer()
    finally:
        gc.set_threshold(*old)
    gc.collect()
    assert ran[0] == 2000
