"""Ops that cut their work into parts give the eager call's bits when they are
captured in a process that has not run them (so that no memory for the parts
is cached): sums along strided dims of doubles that cancel, so that another
order of summation shows; products cut along t; long integer scans.  One graph
holds several of them, which share that memory; replays alternate with eager
work of the same shapes."""
import os
import subprocess
import sys

import pytest

pytestmark = pytest.mark.gpu

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
SCRIPT = r"""
import sys
import numpy as np
sys.path.insert(0, %r)
from pdl_amd import core as C
C.init(0)
rng = np.random.default_rng(11)
kind = sys.argv[1]

def cancelling(rows, cols):
    x = rng.standard_normal((rows // 2, cols)) * 10.0 ** rng.uniform(0, 30, (rows // 2, cols))
    x = np.concatenate([x, -x, rng.standard_normal((rows - rows // 2 * 2, cols))])
    return x[rng.permutation(rows)]

def columns(cols):
    x = C.ndarray.from_numpy(cancelling(30011, cols)).xchg(0, 1)
    return [("sumover", x, [cols]), ("average", x, [cols])]

def product(t, h, k, w):
    a = C.ndarray.from_numpy(rng.standard_normal((h, k)).astype(C.NP_TYPES[t]), t)
    b = C.ndarray.from_numpy(rng.standard_normal((k, w)).astype(C.NP_TYPES[t]), t)
    return [("matmult", a, b, [w, h])]

def scan(t, n):
    x = C.ndarray.from_numpy(rng.integers(-99, 99, (2, n)).astype(C.NP_TYPES[t]), t)
    return [("cumusumover", x, [n, 2])]

ops = {"columns": lambda: columns(6) + columns(24),
       "stepped": lambda: [("dsumover", C.ndarray.from_numpy(cancelling(600001, 1).reshape(-1)).slice((0, 600000, 3)), [])],
       "double": lambda: product(C.L.D, 100, 2000, 90) + product(C.L.D, 70, 3000, 200),
       "float": lambda: product(C.L.F, 100, 2000, 90) + product(C.L.F, 33, 5000, 130),
       "scans": lambda: scan(C.L.L, 100003) + scan(C.L.LL, 70001)}[kind]()
outs = [C.ndarray.new_dense(op[1].dtype, op[-1]) for op in ops]

def body():
    for op, o in zip(ops, outs):
        C._run(op[0], list(op[1:-1]) + [o])

g = C.Graph(body)
for o in outs:
    o.assign(C.ndarray.from_numpy(np.full(o.numpy().shape, 77, C.NP_TYPES[o.dtype]), o.dtype))
g.launch()
C.synchronize()
first = [o.numpy().copy() for o in outs]
body()
eager = [o.numpy().copy() for o in outs]
for op, x, y in zip(ops, first, eager):
    assert x.tobytes() == y.tobytes(), (op[0], x.reshape(-1)[:3], y.reshape(-1)[:3])
for rep in range(3):
    for op, o in zip(ops, outs):
        C._run(op[0], list(op[1:-1]) + [C.ndarray()])
        o.assign(C.ndarray.from_numpy(np.zeros(o.numpy().shape, C.NP_TYPES[o.dtype]), o.dtype))
    g.launch()
    C.synchronize()
    for op, o, y in zip(ops, outs, eager):
        assert o.numpy().tobytes() == y.tobytes(), (rep, op[0])
g.destroy()
body()
for o, y in zip(outs, eager):
    assert o.numpy().tobytes() == y.tobytes()
print("same bits")
""" % ROOT


@pytest.mark.parametrize("kind", ["columns", "stepped", "double", "float", "scans"])
def test_capture_without_an_earlier_run(kind):
    r = subprocess.run([sys.executable, "-c", SCRIPT, kind], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stderr[-3000:]
    assert r.stdout.strip().endswith("same bits")
