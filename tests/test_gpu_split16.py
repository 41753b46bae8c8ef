"""The FP16-split product's ordinary outputs, with 128x128 and 256x256 blocks
(forced through the tuning cache file): ragged sides, inner dimensions from
one pair of slices up, operands unit-stride along either index, an output
through a view, rows over many decades, planted infinities, NaN and
wide-range rows, and replays of a captured product between eager ones.

Every output of finite operands is within 2^-21 |c| + 2^-19 sum |a||b| of the
FP64 product or equals PDL's loop (the PDL-order mode); rows and columns with
a non-finite element equal PDL's loop bit for bit."""
import json
import os
import subprocess
import sys

import pytest

pytestmark = pytest.mark.gpu

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
SHAPES = [(2048, 1024, 2048), (2100, 1030, 2060), (5000, 257, 4100), (1400, 3001, 1900)]
SCRIPT = r"""
import hashlib, json, sys
import numpy as np
sys.path.insert(0, %r)
sys.path.insert(0, %r)
from pdl_amd import core as C
from test_gpu_parity import plant_range_and_nonfinite
C.init(0)
h, t, w = json.loads(sys.argv[1])
rng = np.random.default_rng(h + t)
a = rng.standard_normal((h, t)).astype(np.float32)
a *= np.exp(3.0 * rng.standard_normal((h, 1))).astype(np.float32)
b = rng.standard_normal((t, w)).astype(np.float32)
digests = []
for planted in (False, True):
    if planted:
        marks = plant_range_and_nonfinite(a, b, rng)
    dense = lambda m: C.ndarray.from_numpy(m)
    turned = lambda m: C.ndarray.from_numpy(np.ascontiguousarray(m.T)).xchg(0, 1)
    C.set_matmult_precision("pdlorder")
    pdl = C.matmult(dense(a), dense(b)).numpy()
    C.set_matmult_precision("split16")
    fin = np.outer(np.isfinite(a).all(axis=1), np.isfinite(b).all(axis=0))
    a64, b64 = (np.where(np.isfinite(x), x, 0).astype(np.float64) for x in (a, b))
    truth = a64 @ b64
    bound = 2.0 ** -21 * np.abs(truth) + 2.0 ** -19 * (np.abs(a64) @ np.abs(b64)) + 1e-37
    for name, la, lb in (("dense", dense, dense), ("a turned", turned, dense), ("b turned", dense, turned)):
        x, y = la(a), lb(b)
        d = C.matmult(x, y).numpy()
        bad = fin & ~(np.abs(d.astype(np.float64) - truth) <= bound) & ~(d == pdl)
        assert not bad.any(), (name, planted, np.argwhere(bad)[:5], d[bad][:5], truth[bad][:5])
        if planted:
            for r in marks["nonfinite_rows"]:
                np.testing.assert_array_equal(d[r], pdl[r])
            for col in marks["nonfinite_cols"]:
                np.testing.assert_array_equal(d[:, col], pdl[:, col])
        digests.append(hashlib.sha256(d.tobytes()).hexdigest())
        out = C.ndarray.from_numpy(np.full((w, h), 7, np.float32))
        C._run("matmult", [x, y, out.xchg(0, 1)])
        assert np.ascontiguousarray(out.numpy().T).tobytes() == d.tobytes(), name
    x, y, c = dense(a), dense(b), C.ndarray.new_dense(C.L.F, [w, h])
    C._run("matmult", [x, y, c])
    want = c.numpy().copy()
    g = C.Graph(lambda: C._run("matmult", [x, y, c]))
    other, spare = dense(a[::-1].copy()), C.ndarray.new_dense(C.L.F, [w, h])
    for rep in range(3):
        C._run("matmult", [other, y, spare])
        C._run("mult", [c, C.topdl(0.0), c])
        g.launch()
        C.synchronize()
        assert c.numpy().tobytes() == want.tobytes(), rep
    g.destroy()
out = C.tune_stats()
out["digests"] = digests
print(json.dumps(out))
""" % (ROOT, os.path.join(ROOT, "tests"))

SHORT = r"""
import json, sys
import numpy as np
import torch
sys.path.insert(0, %r)
from pdl_amd import core as C
C.init(0)
h, t, w = json.loads(sys.argv[1])
rng = np.random.default_rng(h + t)
a, b = rng.standard_normal((h, t)).astype(np.float32), rng.standard_normal((t, w)).astype(np.float32)
c = C.matmult(C.ndarray.from_numpy(a), C.ndarray.from_numpy(b))
C.synchronize()

class Seen:
    __cuda_array_interface__ = {"shape": (h, w), "typestr": "<f4", "data": (c._buf.ptr, False), "version": 2}

d = torch.as_tensor(Seen(), device="cuda")
for lo in range(0, h, 1024):    # on the GPU, in FP64, some rows at a time
    x, y = torch.from_numpy(a[lo:lo + 1024]).cuda().double(), torch.from_numpy(b).cuda().double()
    truth = x @ y
    bound = 2.0 ** -21 * truth.abs() + 2.0 ** -19 * (x.abs() @ y.abs()) + 1e-37
    assert bool(((d[lo:lo + 1024].double() - truth).abs() <= bound).all()), lo
out = C.tune_stats()
print(json.dumps(out))
""" % ROOT


def run(script, shape, path):
    env = dict(os.environ, PDLHIP_TUNE_FILE=str(path))
    env.pop("PDLHIP_TUNE", None)
    r = subprocess.run([sys.executable, "-c", script, json.dumps(shape)], env=env, capture_output=True, text=True,
                       timeout=120)
    assert r.returncode == 0, r.stderr[-3000:]
    return json.loads(r.stdout.strip().splitlines()[-1])


def force(path, shape, choice):
    h, t, w = (n.bit_length() - 1 for n in shape)
    path.write_text("matmult:float:ring:h2^%d:w2^%d:t2^%d:gfx950 %d\n" % (h, w, t, choice))


@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "x".join(map(str, s)))
def test_split_product(tmp_path, shape):
    path, digests = tmp_path / "tune.txt", set()
    for choice in (128, 256):
        force(path, shape, choice)
        got = run(SCRIPT, shape, path)
        assert got["measured"] == 0 and got["reused"] >= 1, (choice, got)
        digests.add(tuple(got["digests"][:3]))
    # the layouts and the block shapes pack and sum alike
    assert len(digests) == 1 and len(set(digests.pop())) == 1


@pytest.mark.parametrize("choice", [128, 256])
@pytest.mark.parametrize("t", [32, 33, 65, 97])
def test_few_slices(tmp_path, t, choice):
    path, shape = tmp_path / "tune.txt", (24100, t, 24000)
    force(path, shape, choice)
    got = run(SHORT, shape, path)
    assert got["measured"] == 0 and got["reused"] >= 1, got
