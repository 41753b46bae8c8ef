"""The engine of a float product in the default mode goes by its sizes, and the
block shapes the autotuner may pick within an engine give the same bits: two
products of one shape class in either order, without tuning, with every shape
forced through the tuning cache file, with choices an older file holds, and a
first capture all agree bit for bit."""
import json
import os
import subprocess
import sys

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
# (h, t, w): pairs of one class (the same powers of two), on both sides of the rule
CLASSES = [[(600, 600, 600), (1000, 1000, 1000)], [(520, 40, 700), (1020, 60, 1000)],
           [(1024, 1024, 1024), (2047, 2047, 2047)], [(1030, 1100, 1200), (1999, 1600, 2040)],
           [(1100, 2100, 1100), (2040, 4090, 2030)]]
SCRIPT = r"""
import hashlib, json, sys
import numpy as np
sys.path.insert(0, %r)
from pdl_amd import core as C
C.init(0)
out = {}
for h, t, w in json.loads(sys.argv[1]):
    rng = np.random.default_rng(h + t + w)
    a = C.ndarray.from_numpy(rng.standard_normal((h, t)).astype(np.float32))
    b = C.ndarray.from_numpy(rng.standard_normal((t, w)).astype(np.float32))
    c = C.ndarray.new_dense(C.L.F, [w, h])
    if sys.argv[2] == "capture":
        try:
            g = C.Graph(lambda: C._run("matmult", [a, b, c]))
            g.launch()
            C.synchronize()
            g.destroy()
            out["%%dx%%dx%%d" %% (h, t, w)] = hashlib.sha256(c.numpy().tobytes()).hexdigest()
        except C.PDLError as e:      # the split's packing needs an earlier run
            assert "not cached" in str(e)
        continue
    C._run("matmult", [a, b, c])
    out["%%dx%%dx%%d" %% (h, t, w)] = hashlib.sha256(c.numpy().tobytes()).hexdigest()
print(json.dumps(out))
""" % ROOT


def run(sizes, path, tune=True, how="eager"):
    env = dict(os.environ, PDLHIP_TUNE_FILE=str(path))
    env.pop("PDLHIP_TUNE", None)
    if not tune:
        env["PDLHIP_TUNE"] = "0"
    r = subprocess.run([sys.executable, "-c", SCRIPT, json.dumps(sizes), how], env=env, capture_output=True, text=True,
                       timeout=120)
    assert r.returncode == 0, r.stderr[-3000:]
    return json.loads(r.stdout.strip().splitlines()[-1])


def key(engine, shape):
    return "matmult:float:%s:h2^%d:w2^%d:t2^%d:gfx950" % ((engine,) + tuple(int(np.log2(shape[i])) for i in (0, 2, 1)))


@pytest.mark.parametrize("sizes", CLASSES, ids=["-".join("x".join(map(str, s)) for s in c) for c in CLASSES])
def test_bits_depend_on_sizes_alone(tmp_path, sizes):
    want = run(sizes, tmp_path / "none.txt", tune=False)
    assert run(sizes, tmp_path / "up.txt") == want
    assert run(sizes[::-1], tmp_path / "down.txt") == want
    for choice in (32, 64, 128, 256):
        path = tmp_path / ("forced%d.txt" % choice)
        path.write_text("".join("%s %d\n" % (key(e, s), choice) for e in ("tile", "ring", "tile_or_ring", "default")
                                for s in sizes))
        assert run(sizes, path) == want, choice
    captured = run(sizes, tmp_path / "captured.txt", how="capture")
    assert all(want[k] == v for k, v in captured.items())
