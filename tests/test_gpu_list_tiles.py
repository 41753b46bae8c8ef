"""Matmult lists on the matrix cores at the edges of their tiles and stages:
sides around 16, 32 and 64, inner dimensions from none over less than one
16-byte load and one stage to several, operands unit-stride along either
index, each with 64x64 and 32x32 work items (forced through the tuning cache
file) and in both launch modes.  Every element is held to the bound of any
order of summation: (k + 2) roundings of the sum of the products' sizes."""
import json
import os
import subprocess
import sys

import pytest

pytestmark = pytest.mark.gpu

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
SCRIPT = r"""
import json, sys
import numpy as np
sys.path.insert(0, %r)
from pdl_amd import core as C
C.init(0)
t, layout = int(sys.argv[1]), sys.argv[2]
dt, eps = (np.float32, 2.0 ** -24) if t == C.L.F else (np.float64, 2.0 ** -53)
least = 0 if layout[2:] == "any" else 4
rng = np.random.default_rng(5)
sides, inner = [1, 15, 16, 17, 31, 32, 33, 63, 64, 65, 130], [0, 1, 2, 3, 4, 5, 15, 16, 17, 31, 32, 33, 48, 63, 64, 65, 97, 200]
shapes = [(int(rng.choice(sides)), k, int(rng.choice(sides))) for k in inner for _ in range(6) if k >= least]

def operand(rows, cols, transposed):
    x = rng.standard_normal((cols, rows) if transposed else (rows, cols)).astype(dt)
    nd = C.ndarray.from_numpy(x, t)
    return (x.T, nd.xchg(0, 1)) if transposed else (x, nd)

a = [operand(h, k, layout[0] == "t") for h, k, w in shapes]
b = [operand(k, w, layout[1] == "t") for h, k, w in shapes]
ml = C.MatmultList([x[1] for x in a], [x[1] for x in b])
worst, launches = 0.0, []
for mode in ("queue", "each"):
    for o in ml.outputs:
        o.assign(C.ndarray.from_numpy(np.full(o.numpy().shape, np.nan, dt), t))
    ml.launch(mode)
    outs = [o.numpy() for o in ml.outputs]
    launches.append(outs)
    for (h, k, w), (x, _), (y, _), o in zip(shapes, a, b, outs):
        x, y = x.astype(np.longdouble), y.astype(np.longdouble)
        assert o.shape == (h, w)
        over = np.abs(o - x @ y) - (k + 2) * eps * (np.abs(x) @ np.abs(y))
        assert not np.isnan(over).any(), (mode, h, k, w)
        worst = max(worst, float(over.max()))
same = all(np.array_equal(x, y) for x, y in zip(*launches))
ml.free()
out = C.tune_stats()
out.update({"worst": worst, "same": same})
print(json.dumps(out))
""" % ROOT


def run(env, t, layout):
    r = subprocess.run([sys.executable, "-c", SCRIPT, str(t), layout], env=env, capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stderr[-3000:]
    return json.loads(r.stdout.strip().splitlines()[-1])


@pytest.mark.parametrize("t", [9, 10], ids=["float", "double"])
@pytest.mark.parametrize("layout", ["nnany", "nn", "tn", "nt", "tt"])
def test_list_tile_edges(tmp_path, t, layout):
    path = tmp_path / "tune.txt"
    env = dict(os.environ, PDLHIP_TUNE_FILE=str(path))
    env.pop("PDLHIP_TUNE", None)
    run(env, t, layout)
    keys = [line.split()[0] for line in path.read_text().splitlines() if line.startswith("list:")]
    assert len(keys) == 1, keys
    for c in (0, 2):
        path.write_text("%s %d\n" % (keys[0], c))
        got = run(env, t, layout)
        assert got["measured"] == 0 and got["reused"] >= 1, (c, got)
        assert got["worst"] <= 0 and got["same"], (c, got)
