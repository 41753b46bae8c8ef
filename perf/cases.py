"""Work that programs give this package, for timing: eager expressions from a
few elements up, image arithmetic over mixed types, broadcasts through
transposed and dummy views, statistics along rows and along columns, scans,
bad values, single / batched / listed matrix products, and ragged lists
replayed as a graph.

listed() names a dozen sizes, draw() gives others of the same ranges,
prepare() makes what a program holds before the call (inputs in HBM, prepared
lists, chains and graphs), run() is one pass, work() the bytes and operations
that a pass cannot do without, exact() the results in 64 bits by plain torch.

Dims are written in PDL's order (dim 0 fastest); a tensor of an ndarray has
them reversed."""
import math

import numpy as np
import torch

from pdl_amd import core as C

TORCH = {C.L.B: torch.uint8, C.L.S: torch.int16, C.L.L: torch.int32, C.L.LL: torch.int64, C.L.IND: torch.int64,
         C.L.F: torch.float32, C.L.D: torch.float64}
TYPESTR = {C.L.B: "|u1", C.L.S: "<i2", C.L.US: "<i2", C.L.L: "<i4", C.L.LL: "<i8", C.L.IND: "<i8", C.L.F: "<f4",
           C.L.D: "<f8"}


# ---------------------------------------------------------------- the cases
def listed():
    return [
        # a Perl-level expression over a small table: a handful of launches, latency only
        {"name": "expr_f64_48x50", "kind": "expr", "dtype": "f64", "nx": 48, "ny": 50, "fused": False},
        # c = a*b + a with s = sumover(c) over a mid-size array, as one prepared fused chain
        {"name": "chain_f64_2048", "kind": "expr", "dtype": "f64", "nx": 2048, "ny": 2048, "fused": True},
        # reducing a detector frame: ushort counts, float dark and flat frames, byte mask, whole-frame statistics
        {"name": "calib_2149x2047", "kind": "calib", "nx": 2149, "ny": 2047},
        # a gain per row over a stack of transposed frames, then the statistics of each row
        {"name": "broadcast_f32_4096x16", "kind": "broadcast", "dtype": "f32", "nx": 4096, "ny": 4096, "nk": 16},
        # column statistics of a long table
        {"name": "columns_f32_24x1000003", "kind": "columns", "dtype": "f32", "ncol": 24, "nrow": 1000003},
        # running and total counts of many channels
        {"name": "scan_i32_4096", "kind": "scan", "dtype": "i32", "n": 4096, "rows": 4096},
        # short samples with 1% missing: sums and counts of the good ones, and the missing ones filled
        {"name": "bad_i16_8192", "kind": "bad", "n": 8192, "rows": 8192},
        # large single product, the default float precision
        {"name": "matmult_f32_8192", "kind": "matmult", "dtype": "f32", "t": 8192, "h": 8192, "w": 8192},
        # the matrix_multiplication benchmark's size, double
        {"name": "matmult_f64_1500", "kind": "matmult", "dtype": "f64", "t": 1500, "h": 1500, "w": 1500},
        # many small products by broadcasting
        {"name": "batch_f32_64x65536", "kind": "batch", "dtype": "f32", "t": 64, "h": 64, "w": 64, "count": 65536},
        # many products of uneven sizes, as a prepared list
        {"name": "list_f32_4096", "kind": "list", "dtype": "f32", "count": 4096, "lo": 8, "hi": 256},
        # vectors of uneven lengths: a weighted, masked sum of squares and a running sum of each, as a graph
        {"name": "ragged_40000", "kind": "ragged", "nvec": 40000},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["expr", "expr", "calib", "broadcast", "columns", "scan", "bad", "matmult", "matmult", "batch",
                       "list", "ragged"])
    if kind == "expr":
        return {"kind": kind, "dtype": rng.choice(["f32", "f64"]), "nx": _log(rng, 1, 2600), "ny": _log(rng, 1, 2600),
                "fused": rng.random() < 0.5}
    if kind == "calib":
        return {"kind": kind, "nx": _log(rng, 100, 6000), "ny": _log(rng, 100, 6000)}
    if kind == "broadcast":
        return {"kind": kind, "dtype": rng.choice(["f32", "f64"]), "nx": _log(rng, 100, 4096), "ny": _log(rng, 100, 4096),
                "nk": _log(rng, 1, 8)}
    if kind == "columns":
        ncol = _log(rng, 2, 1000000)
        return {"kind": kind, "dtype": rng.choice(["f32", "f64"]), "ncol": ncol,
                "nrow": _log(rng, 8, max(16, min(1000000, 60000000 // ncol)))}
    if kind == "scan":
        n = _log(rng, 16, 1000000)
        return {"kind": kind, "dtype": rng.choice(["i32", "i32", "i64", "f32", "f64"]), "n": n,
                "rows": _log(rng, 1, max(2, min(100000, 16000000 // n)))}
    if kind == "bad":
        n = _log(rng, 64, 100000)
        return {"kind": kind, "n": n, "rows": _log(rng, 16, max(32, min(100000, 67000000 // n)))}
    if kind == "matmult":
        dtype = rng.choice(["f32", "f64"])
        hi = 6000 if dtype == "f32" else 3000
        return {"kind": kind, "dtype": dtype, "t": _log(rng, 16, hi), "h": _log(rng, 16, hi), "w": _log(rng, 16, hi)}
    if kind == "batch":
        t, h, w = (_log(rng, 4, 128) for _ in range(3))
        return {"kind": kind, "dtype": rng.choice(["f32", "f64"]), "t": t, "h": h, "w": w,
                "count": _log(rng, 64, max(128, min(65536, 100000000 // max(t * h, t * w, h * w))))}
    if kind == "list":
        lo = _log(rng, 2, 64)
        return {"kind": kind, "dtype": rng.choice(["f32", "f64"]), "count": _log(rng, 16, 4096), "lo": lo,
                "hi": _log(rng, lo + 1, 256)}
    return {"kind": kind, "nvec": _log(rng, 100, 40000)}


# ---------------------------------------------------------------- ndarrays and tensors
class _Seen:
    """an ndarray's whole buffer as torch takes foreign device memory in"""

    def __init__(self, x):
        self.x = x
        self.__cuda_array_interface__ = {"shape": tuple(x.dims[::-1]), "typestr": TYPESTR[x.dtype],
                                         "data": (x._buf.ptr, False), "version": 2}


def tensor(x):
    """a dense ndarray as a tensor over the same memory, which it keeps alive"""
    return torch.as_tensor(_Seen(x), device="cuda")


def ndarray(t, dtype):
    """a new ndarray with the values of tensor t (a device copy)"""
    x = C.ndarray.new_dense(dtype, list(t.shape[::-1]))
    tensor(x).copy_(t)
    return x


def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _code(case):
    return {"f32": C.L.F, "f64": C.L.D, "i32": C.L.L, "i64": C.L.LL}[case["dtype"]]


def _uniform(g, *shape, dtype=torch.float32):
    return torch.rand(shape, generator=g, device="cuda", dtype=dtype) * 2 - 1


def _normal(g, *shape, dtype=torch.float32):
    return torch.randn(shape, generator=g, device="cuda", dtype=dtype)


def _lengths(case):
    """the vectors' lengths, lognormal(8, 1.5) from 1 to 2^20"""
    r = np.random.RandomState(case["nvec"])
    return np.clip(np.round(np.exp(8.0 + 1.5 * r.standard_normal(case["nvec"]))), 1, 2 ** 20).astype(np.int64)


def _sides(case):
    """the listed products' sides, uniform in lo..hi"""
    return np.random.RandomState(case["count"]).randint(case["lo"], case["hi"] + 1, case["count"]).astype(np.int64)


def _starts(sizes):
    return np.concatenate([[0], np.cumsum(sizes)[:-1]]).astype(np.int64)


def inputs(case, seed):
    """the case's inputs as tensors on the GPU"""
    g, k = _gen(seed), case["kind"]
    if k == "expr":
        d = TORCH[_code(case)]
        return [_uniform(g, case["ny"], case["nx"], dtype=d) for _ in range(2)]
    if k == "calib":
        s = (case["ny"], case["nx"])
        raw = torch.randint(100, 30000, s, generator=g, device="cuda", dtype=torch.int16)
        dark = 100 + 3 * _normal(g, *s)
        flat = 1 + 0.1 * _uniform(g, *s)
        mask = (torch.rand(s, generator=g, device="cuda") < 0.98).to(torch.uint8)
        return [raw, dark, flat, mask]
    if k == "broadcast":
        d = TORCH[_code(case)]
        return [_normal(g, case["nk"], case["ny"], case["nx"], dtype=d), _normal(g, case["nk"], case["ny"], dtype=d)]
    if k == "columns":
        return [_normal(g, case["nrow"], case["ncol"], dtype=TORCH[_code(case)])]
    if k == "scan":
        s = (case["rows"], case["n"])
        if case["dtype"][0] == "f":
            return [_uniform(g, *s, dtype=TORCH[_code(case)])]
        return [torch.randint(-2 ** 20, 2 ** 20 + 1, s, generator=g, device="cuda", dtype=TORCH[_code(case)])]
    if k == "bad":
        s = (case["rows"], case["n"])
        v = torch.randint(-32767, 32768, s, generator=g, device="cuda", dtype=torch.int16)
        v[torch.rand(s, generator=g, device="cuda") < 0.01] = -32768
        return [v]
    if k == "matmult":
        d = TORCH[_code(case)]
        return [_normal(g, case["h"], case["t"], dtype=d), _normal(g, case["t"], case["w"], dtype=d)]
    if k == "batch":
        d, n = TORCH[_code(case)], case["count"]
        return [_uniform(g, n, case["h"], case["t"], dtype=d), _uniform(g, n, case["t"], case["w"], dtype=d)]
    if k == "list":
        tot = int((_sides(case) ** 2).sum())
        return [_uniform(g, tot, dtype=TORCH[_code(case)]) for _ in range(2)]
    tot = int(_lengths(case).sum())
    return [_normal(g, tot), _normal(g, tot), torch.rand(tot, generator=g, device="cuda"),
            torch.randint(0, 2, (tot,), generator=g, device="cuda", dtype=torch.uint8),
            torch.randint(-2 ** 40, 2 ** 40, (tot,), generator=g, device="cuda", dtype=torch.int64)]


# ---------------------------------------------------------------- what a program holds, and one pass
def prepare(case, seed):
    C.init(0)
    k, ins = case["kind"], inputs(case, seed)
    torch.cuda.synchronize()
    s = {"kind": k}
    if k == "expr":
        t = _code(case)
        a, b = (ndarray(x, t) for x in ins)
        s.update(a=a, b=b)
        if case["fused"]:
            c, r = C.ndarray.new_dense(t, a.dims), C.ndarray.new_dense(t, a.dims[1:])
            s["chain"] = C.Chain([a, b], [("mult", 0, 1), ("plus", ("node", 0), 0)], "sumover", value=c, result=r)
            s["out"] = (tensor(c), tensor(r))
    elif k == "calib":
        s.update(raw=ndarray(ins[0], C.L.US), dark=ndarray(ins[1], C.L.F), flat=ndarray(ins[2], C.L.F),
                 mask=ndarray(ins[3], C.L.B))
    elif k == "broadcast":
        t = _code(case)
        s.update(x=ndarray(ins[0], t), y=ndarray(ins[1], t))
    elif k in ("columns", "scan"):
        s["x"] = ndarray(ins[0], _code(case))
    elif k == "bad":
        s["x"] = ndarray(ins[0], C.L.S)
        s["x"].badflag(True)
    elif k in ("matmult", "batch"):
        t = _code(case)
        s.update(a=ndarray(ins[0], t), b=ndarray(ins[1], t))
    elif k == "list":
        t, sides = _code(case), _sides(case)
        starts = _starts(sides ** 2)
        a, b = ndarray(ins[0], t), ndarray(ins[1], t)
        c = C.ndarray.new_dense(t, a.dims)
        views = [[C.view_into(p, [int(n), int(n)], int(o)) for n, o in zip(sides, starts)] for p in (a, b, c)]
        s["list"], s["out"] = C.MatmultList(*views), tensor(c)
    else:
        lens = _lengths(case)
        starts = _starts(lens)
        a, b, w = (ndarray(x, C.L.F) for x in ins[:3])
        m, v = ndarray(ins[3], C.L.B), ndarray(ins[4], C.L.LL)
        two = C.topdl(2)
        sums, runs = C.ndarray.new_dense(C.L.F, [case["nvec"]]), C.ndarray.new_dense(C.L.LL, v.dims)
        cut = lambda p: [C.view_into(p, [int(n)], int(o)) for n, o in zip(lens, starts)]  # noqa: E731
        total = C.Ragged([[x, y, two, z, q] for x, y, z, q in zip(cut(a), cut(b), cut(w), cut(m))],
                         [("minus", 0, 1), ("power", ("node", 0), 2), ("mult", ("node", 1), 3), ("mult", ("node", 2), 4)],
                         "sumover", outputs=[C.view_into(sums, [], i) for i in range(case["nvec"])])
        running = C.Ragged([[x] for x in cut(v)], [], "cumusumover", outputs=cut(runs))
        s["held"] = (total, running)
        s["graph"] = C.Graph(lambda: (total.run(), running.run()))
        s["out"] = (tensor(sums), tensor(runs))
    torch.cuda.synchronize()
    return s


def run(s):
    k = s["kind"]
    if k == "expr":
        if "chain" in s:
            s["chain"].run()
            return s["out"]
        c = s["a"] * s["b"] + s["a"]
        return tensor(c), tensor(c.sumover())
    if k == "calib":
        img = (s["raw"] - s["dark"]) / s["flat"] * s["mask"]
        lo, hi = img.minmax()
        return tensor(img), tensor(img.avg()), tensor(lo), tensor(hi)
    if k == "broadcast":
        z = s["x"].xchg(0, 1) * s["y"].dummy(1)
        return tensor(z), tensor(z.sumover()), tensor(z.average()), tensor(z.minimum()), tensor(z.maximum())
    if k == "columns":
        v = s["x"].xchg(0, 1)
        return tensor(v.average()), tensor(v.minimum()), tensor(v.maximum())
    if k == "scan":
        return tensor(s["x"].sumover()), tensor(s["x"].cumusumover())
    if k == "bad":
        v = s["x"]
        return tensor(v.sumover()), tensor(v.isgood().sumover()), tensor(v.setbadtoval(0))
    if k in ("matmult", "batch"):
        return tensor(C.matmult(s["a"], s["b"]))
    if k == "list":
        s["list"].launch()
        return s["out"]
    s["graph"].launch()
    return s["out"]


# ---------------------------------------------------------------- what a pass cannot do without
def work(case):
    k = case["kind"]
    e = {"f32": 4, "f64": 8, "i32": 4, "i64": 8}.get(case.get("dtype"), 0)
    if k == "expr":
        n = case["nx"] * case["ny"]
        return {"bytes": (3 * n + case["ny"]) * e, "flops": 3 * n}
    if k == "calib":
        n = case["nx"] * case["ny"]
        return {"bytes": n * (2 + 4 + 4 + 1 + 4) + 12, "flops": 6 * n}
    if k == "broadcast":
        n, o = case["nx"] * case["ny"] * case["nk"], case["nx"] * case["nk"]
        return {"bytes": (2 * n + case["ny"] * case["nk"] + 4 * o) * e, "flops": 5 * n}
    if k == "columns":
        n = case["ncol"] * case["nrow"]
        return {"bytes": (n + 3 * case["ncol"]) * e, "flops": 3 * n}
    if k == "scan":
        n = case["n"] * case["rows"]
        return {"bytes": (2 * n + case["rows"]) * e, "flops": 2 * n}
    if k == "bad":
        n = case["n"] * case["rows"]
        return {"bytes": 4 * n + 8 * case["rows"], "flops": 3 * n}
    if k in ("matmult", "batch"):
        t, h, w, n = case["t"], case["h"], case["w"], case.get("count", 1)
        return {"bytes": n * (t * h + t * w + h * w) * e, "flops": 2 * n * t * h * w}
    if k == "list":
        n = _sides(case).astype(np.float64)
        return {"bytes": float(3 * (n ** 2).sum() * e), "flops": float(2 * (n ** 3).sum())}
    tot = int(_lengths(case).sum())
    return {"bytes": tot * (4 + 4 + 4 + 1 + 8 + 8) + 4 * case["nvec"], "flops": 6 * tot}


# ---------------------------------------------------------------- the results in 64 bits
def exact(case, seed):
    k, ins = case["kind"], inputs(case, seed)
    if k == "expr":
        a, b = (x.double() for x in ins)
        c = a * b + a
        return c, c.sum(1)
    if k == "calib":
        raw, dark, flat, mask = (x.double() for x in ins)
        img = (raw - dark) / flat * mask
        return img, img.mean(), img.min(), img.max()
    if k == "broadcast":
        z = ins[0].double().transpose(1, 2).contiguous() * ins[1].double()[:, None, :]
        # a row of z is one x over all y: its values lie along y
        return z, z.sum(2), z.mean(2), z.amin(2), z.amax(2)
    if k == "columns":
        x = ins[0].double()
        return x.mean(0), x.amin(0), x.amax(0)
    if k == "scan":
        x = ins[0]
        if case["dtype"][0] == "f":
            x = x.double()
            return x.sum(1), x.cumsum(1)
        return x.sum(1, dtype=torch.int64).to(x.dtype), x.cumsum(1, dtype=torch.int64).to(x.dtype)
    if k == "bad":
        v = ins[0]
        good = v != -32768
        return (torch.where(good, v, 0).sum(1, dtype=torch.int32), good.sum(1, dtype=torch.int32),
                torch.where(good, v, 0).to(torch.int16))
    if k == "matmult":
        return ins[0].double() @ ins[1].double()
    if k == "batch":
        return torch.cat([torch.bmm(a.double(), b.double()) for a, b in zip(ins[0].split(4096), ins[1].split(4096))])
    if k == "list":
        a, b = (x.double().cpu() for x in ins)
        sides = _sides(case)
        return torch.cat([(a[o:o + n * n].view(n, n) @ b[o:o + n * n].view(n, n)).reshape(-1)
                          for n, o in zip(map(int, sides), map(int, _starts(sides ** 2)))])
    a, b, w = (x.double() for x in ins[:3])
    z = (a - b) ** 2 * w * ins[3].double()
    lens = torch.from_numpy(_lengths(case)).cuda()
    sums = torch.segment_reduce(z, "sum", lengths=lens)
    # a vector's running sum: the list's, less what ran up before its start (64-bit sums wrap, so this is exact)
    ran = ins[4].cumsum(0)
    before = torch.cat([ran.new_zeros(1), ran])[lens.cumsum(0) - lens]
    return sums, ran - torch.repeat_interleave(before, lens)
