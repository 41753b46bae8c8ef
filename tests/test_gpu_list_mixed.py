"""Matmult lists whose products do not all load alike: inner dimensions from
none to less than one 16-byte load, and transposed operands, among dense
products, few or many of them.  Both work item sizes (forced through the
tuning cache file), both launch modes and replays of a captured launch;
outputs within the bound of any order of summation, and in the bits they have
in a list of their own kind."""
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
t, kind = int(sys.argv[1]), sys.argv[2]
dt, eps = (np.float32, 2.0 ** -24) if t == C.L.F else (np.float64, 2.0 ** -53)
rng = np.random.default_rng(7)
many = 6 if len(sys.argv) > 3 else 400       # below and above the size from which the parts have a launch each
plain = [(int(h), int(k), int(w), "nn") for h, k, w in rng.integers(4, 150, (many, 3))]
odd = {"one short": [(70, 1, 65, "nn")],
       "short": [(int(rng.integers(1, 140)), k, int(rng.integers(1, 140)), "nn") for k in (0, 1, 2, 3) for _ in range(5)],
       "layouts": [(int(h), int(k), int(w), lay) for lay in ("tn", "nt", "tt") for h, k, w in rng.integers(4, 150, (6, 3))],
       "mostly short": [(int(rng.integers(1, 140)), k, int(rng.integers(1, 140)), "nn") for k in (1, 2, 3) for _ in range(60)],
       "only empty": [(9, 0, 70, "nn")]}[kind]
if kind == "only empty":
    plain = plain[:1]
shapes = plain + odd
shapes = [shapes[i] for i in rng.permutation(len(shapes))]

def operand(rows, cols, transposed):
    x = rng.standard_normal((cols, rows) if transposed else (rows, cols)).astype(dt)
    nd = C.ndarray.from_numpy(x, t)
    return (x.T, nd.xchg(0, 1)) if transposed else (x, nd)

a = [operand(h, k, lay[0] == "t") for h, k, w, lay in shapes]
b = [operand(k, w, lay[1] == "t") for h, k, w, lay in shapes]
ml = C.MatmultList([x[1] for x in a], [x[1] for x in b])

def wipe(l):
    for o in l.outputs:
        o.assign(C.ndarray.from_numpy(np.full(o.numpy().shape, np.nan, dt), t))

got = {}
graph = C.Graph(lambda: ml.launch("queue"))
for mode in ("queue", "each", "graph", "graph again"):
    wipe(ml)
    if mode.startswith("graph"):
        graph.launch()
        C.synchronize()
    else:
        ml.launch(mode)
    got[mode] = [o.numpy().copy() for o in ml.outputs]
worst = 0.0
for s, (x, _), (y, _), o in zip(shapes, a, b, got["queue"]):
    x, y = x.astype(np.longdouble), y.astype(np.longdouble)
    over = np.abs(o - x @ y) - (s[1] + 2) * eps * (np.abs(x) @ np.abs(y))
    assert o.shape == (s[0], s[2]) and not np.isnan(over).any(), s
    worst = max(worst, float(over.max()))
same = all(p.tobytes() == q.tobytes() for m in got for p, q in zip(got["queue"], got[m]))
graph.destroy()
for lay in ("nn", "tn"):
    pick = [i for i, s in enumerate(shapes) if s[3] == lay and s[1] >= 4]
    if not pick:
        continue
    alone = C.MatmultList([a[i][1] for i in pick], [b[i][1] for i in pick])
    alone.launch("queue" if lay == "nn" else "each")
    same = same and all(o.numpy().tobytes() == got["queue"][i].tobytes() for i, o in zip(pick, alone.outputs))
    alone.free()
ml.free()
out = C.tune_stats()
out.update({"worst": worst, "same": same})
print(json.dumps(out))
""" % ROOT


def run(env, t, kind, *few):
    r = subprocess.run([sys.executable, "-c", SCRIPT, str(t), kind, *few], env=env, capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stderr[-3000:]
    return json.loads(r.stdout.strip().splitlines()[-1])


@pytest.mark.parametrize("t", [9, 10], ids=["float", "double"])
@pytest.mark.parametrize("kind", ["one short", "short", "layouts", "mostly short", "only empty"])
def test_mixed_lists(tmp_path, t, kind):
    path = tmp_path / "tune.txt"
    env = dict(os.environ, PDLHIP_TUNE_FILE=str(path))
    env.pop("PDLHIP_TUNE", None)
    for few in ([], ["few"]):
        run(env, t, kind, *few)
        keys = [line.split()[0] for line in path.read_text().splitlines() if line.startswith("list:")]
        for c in (0, 2):
            path.write_text("".join("%s %d\n" % (k, c) for k in keys))
            got = run(env, t, kind, *few)
            assert got["measured"] == 0 and got["reused"] >= 1, (c, got)
            assert got["worst"] <= 0 and got["same"], (c, got)
        path.unlink()
